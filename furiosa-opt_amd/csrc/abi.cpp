// The C ABI (include/furiosa_hip.h): handle management, error translation, and the host-side
// planning that turns each Backend seam call's mappings into kernel descriptors.
#include <algorithm>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "runtime.hpp"

using namespace fo;
namespace fm = fo::mapping;

// The no-alloc entry point's working memory (fo_contraction_noalloc): one array per GPU, resident
// from the library's first use on that GPU until the process ends. In host code `scratch` only
// names the symbol; its device address comes from hipGetSymbolAddress (static_scratch_init).
constexpr uint64_t kStaticScratchBytes = 64ull << 20;
static __device__ __align__(256) uint8_t scratch[kStaticScratchBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_static_scratch_mu;
void* g_static_scratch[kMaxDevices] = {};

// Resolves `scratch` on the current device (`device`) once; called by fo_runtime_init.
void static_scratch_init(int device) {
  require(device >= 0 && device < kMaxDevices, "device index beyond the static scratch table");
  std::lock_guard<std::mutex> lock(g_static_scratch_mu);
  if (g_static_scratch[device]) return;
  void* p = nullptr;
  FO_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  require(p != nullptr, "static scratch: no device address");
  g_static_scratch[device] = p;
}

// The device address of `scratch` on the runtime's GPU, checked against the request.
void* static_scratch(const fo_runtime* rt, uint64_t bytes, const char* what) {
  require(bytes <= kStaticScratchBytes, std::string(what) + ": needs " + std::to_string(bytes) +
                                            " bytes of scratch, more than the " +
                                            std::to_string(kStaticScratchBytes >> 20) + " MiB static scratch");
  void* p = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_static_scratch_mu);
    p = g_static_scratch[rt->device];
  }
  require(p != nullptr, "static scratch not resolved for this device (fo_runtime_init resolves it)");
  return p;
}

thread_local std::string g_last_error;

}  // namespace

void fo_pool::release(void* ptr, uint64_t capacity) {
  {
    std::lock_guard<std::mutex> lock(mu);
    if (!orphaned && cached_bytes + capacity <= kMaxCached) {
      cached.emplace(capacity, ptr);
      cached_bytes += capacity;
      return;
    }
  }
  (void)hipSetDevice(device);
  (void)hipDeviceSynchronize();
  (void)hipFree(ptr);
}

namespace {

// Pending casts. The engine widens both contraction operands with Backend::map before
// contraction_prewidened (contract_outer, engine/contraction/outer/mod.rs:145-163), so a
// contraction over f32 (i32) operands usually reads buffers that are exact casts of bf16 or 8-bit
// float (i8) data. fo_map records each such cast (dst, src, source type, element count) and defers
// the cast itself: a contraction whose two operands both have a record of the same source type
// reads the narrow sources instead and never needs the wide copy. The GEMV and the generic folds
// widen them the same way the map would, so their results are those of the wide copies bit for
// bit; the MFMA kernels (both free extents at least 8 on an MFMA-able layout) consume them directly
// and sum each cell in another order, so an f32 result from them is held to the contraction
// tolerance, not to the fold's bits (i32 results stay exact). The engine's kernels also round f32 results to bf16 and widen them back before the next
// f32 step (a narrow, then a widen); the f32 -> bf16 cast is deferred the same way, and a zip, map
// or reduce that reads such a widen reads the f32 data and rounds it on load. Any other use of a
// buffer with a deferred cast into it (check_buf) runs the cast first (and the cast into its source
// before it), on the stream of the runtime that issued it; so does a write to its source
// (note_write), before the source changes. A write to either side drops the record. A source freed
// by its owner while a record reads it is kept (retired) until no record reads it, so an engine
// that narrows into a temporary, widens it and drops the temporary still has both casts deferred.
// Records are process-wide, as buffers are.
struct WidenRecord {
  const fo_buffer* dst;
  const fo_buffer* src;
  fo_dtype src_t;
  uint64_t n;
  fo_dtype dst_t;
  fo_op op;
  fo_runtime* rt;  // the runtime whose stream the deferred cast goes on
  bool deferred;   // the cast has not run yet
  // A broadcast (kind 1) instead of a cast: a transpose over the whole of the f32 dst whose src
  // digits form one contiguous run, dst[i] = src[(i / div) % mod] for i < n; `wheels` launch it.
  int kind = 0;
  uint32_t div = 1, mod = 1;
  Wheels<1> wheels{};
  // A chain of f32 -> f32 maps (kind 2) instead of a cast: dst = pre.op[pre.n - 1](... pre.op[0](src)).
  PreOps pre{};
  // A relayout (kind 3) instead of a cast: the full-view transposes views[0] -> views[1] -> ... of
  // elements of type xt, as consecutive Tensor::transpose calls into fresh storages make them, in the
  // direct form (one transpose views[0] -> views.back(): `wheels`, `count` positions of dst).
  std::vector<std::string> views;
  fo_dtype xt = FO_I8;
  int64_t count = 0;
};
std::mutex g_widen_mu;
std::vector<WidenRecord> g_widen;
std::vector<fo_buffer*> g_retired;  // freed by their owners, kept while a record reads them

bool is_narrow(const WidenRecord& r) { return r.kind == 0 && r.src_t == FO_F32 && r.dst_t == FO_BF16; }
bool is_bcast(const WidenRecord& r) { return r.kind == 1; }
bool is_chain(const WidenRecord& r) { return r.kind == 2; }
bool is_xpose(const WidenRecord& r) { return r.kind == 3; }

// A buffer's block leaves it (the buffer is being freed, rec the recording open at that moment or
// none), then the buffer goes. A block freed while recording stays with the recording's memory,
// since the graph may touch it; later allocations of the recording reuse it unless an earlier graph
// owns it.
void free_block(fo_buffer* buf, const std::shared_ptr<fo_graph_mem>& rec) {
  if (buf->pool) {
    std::lock_guard<std::mutex> lock(buf->pool->mu);
    buf->pool->unfilled.erase(buf);
  }
  if (buf->ptr) {
    if (rec) {
      if (buf->graph_mem == rec) {
        rec->reuse.emplace(buf->capacity, buf->ptr);
      } else if (buf->graph_mem) {
        rec->keep.push_back(buf->graph_mem);
      } else {
        rec->blocks.emplace_back(buf->capacity, buf->ptr);
        rec->reuse.emplace(buf->capacity, buf->ptr);
      }
    } else if (!buf->graph_mem) {
      if (buf->pool) {
        buf->pool->release(buf->ptr, buf->capacity);
      } else {
        (void)hipSetDevice(buf->device);
        (void)hipDeviceSynchronize();
        (void)hipFree(buf->ptr);
      }
    }  // else the block is its recording's, returned when that memory's last holder goes
  }
  delete buf;
}

// Erases the records that match, then lets go of retired buffers that no record reads any more
// (dropping the records that cast into them, which nothing can read now, and so on); returns those
// buffers, for the caller to free once any cast that reads them has been launched. Lock held.
template <typename Pred>
std::vector<fo_buffer*> erase_records(Pred drop) {
  g_widen.erase(std::remove_if(g_widen.begin(), g_widen.end(), drop), g_widen.end());
  std::vector<fo_buffer*> gone;
  for (bool changed = true; changed;) {
    changed = false;
    for (size_t i = 0; i < g_retired.size(); ++i) {
      fo_buffer* b = g_retired[i];
      if (std::any_of(g_widen.begin(), g_widen.end(), [b](const WidenRecord& r) { return r.src == b; })) continue;
      g_widen.erase(std::remove_if(g_widen.begin(), g_widen.end(), [b](const WidenRecord& r) { return r.dst == b; }),
                    g_widen.end());
      gone.push_back(b);
      g_retired.erase(g_retired.begin() + (std::ptrdiff_t)i);
      changed = true;
      break;
    }
  }
  return gone;
}

// Records being run (run_deferred) are copies that still point at their buffers, and running one
// can drop the records of others (a source's own cast runs first, then run records go), which may
// let a retired source go. So while any run is in progress, retired buffers that lose their last
// reader are held here and freed when the outermost run has launched everything it copied.
std::mutex g_free_mu;
int g_run_depth = 0;
std::vector<fo_buffer*> g_free_later;

void free_now(const std::vector<fo_buffer*>& gone) {
  for (fo_buffer* b : gone) {
    std::shared_ptr<fo_graph_mem> rec = std::move(b->retired_in);
    free_block(b, rec);
  }
}

void free_retired(const std::vector<fo_buffer*>& gone) {
  if (gone.empty()) return;
  {
    std::lock_guard<std::mutex> lock(g_free_mu);
    if (g_run_depth > 0) {
      g_free_later.insert(g_free_later.end(), gone.begin(), gone.end());
      return;
    }
  }
  free_now(gone);
}

// Marks a run of deferred records in progress for its lifetime (see free_retired).
struct RunScope {
  RunScope() {
    std::lock_guard<std::mutex> lock(g_free_mu);
    ++g_run_depth;
  }
  ~RunScope() {
    std::vector<fo_buffer*> gone;
    {
      std::lock_guard<std::mutex> lock(g_free_mu);
      if (--g_run_depth == 0) gone.swap(g_free_later);
    }
    try {
      free_now(gone);
    } catch (...) {  // a failed free leaves its error for the next call to report
    }
  }
};

void materialize(const fo_buffer* b);
void fill_pending(fo_runtime* rt, const fo_buffer* b);
void mark_filled(fo_buffer* b);

// One op's trace span: events recorded on the runtime's stream before and after its launches.
struct TraceScope {
  fo_runtime* rt;
  const char* name;
  hipEvent_t begin = nullptr;
  TraceScope(fo_runtime* r, const char* n) : rt(r), name(n) {
    if (!rt->trace_sink) return;
    FO_HIP(hipEventCreate(&begin));
    FO_HIP(hipEventRecord(begin, rt->stream));
  }
  ~TraceScope() {
    if (!begin) return;
    hipEvent_t end = nullptr;
    if (hipEventCreate(&end) == hipSuccess && hipEventRecord(end, rt->stream) == hipSuccess) {
      rt->spans.push_back({name, begin, end});
    } else {
      (void)hipEventDestroy(begin);
      if (end) (void)hipEventDestroy(end);
    }
  }
};


// Runs deferred casts, in order, outside the lock; a cast whose source has a deferred cast into it
// runs that one first.
void run_deferred(const std::vector<WidenRecord>& rs) {
  RunScope running;  // no buffer a copied record points at is freed before the loop ends
  for (auto& r : rs) {
    materialize(r.src);
    FO_HIP(hipSetDevice(r.rt->device));
    if (is_bcast(r)) {
      launch_relayout(r.rt->stream, r.dst->ptr, r.src->ptr, 4, 0, 0, (int64_t)r.n, r.wheels);
    } else if (is_xpose(r)) {
      TraceScope span(r.rt, "transpose");  // the recorded op's own span, when it runs
      fo_buffer* d = const_cast<fo_buffer*>(r.dst);
      const int64_t eb = dtype_bytes(r.xt);
      const uint64_t cap = (d->capacity + 15) & ~15ull;  // the bytes a zero fill would clear
      if (d->zero_pending && cap % (uint64_t)eb == 0 && cap / (uint64_t)eb < (1ull << 31)) {
        // A fresh storage the views leave partly dead (a padded slice or cluster layout): one pass
        // writes the live cells from the source and zero everywhere else the fill would have,
        // instead of the fill and then the relayout.
        Chain c;
        c.n = 1;
        c.zero_unwritten = 1;
        c.total = (uint32_t)(cap / (uint64_t)eb);
        c.step[0] = ChainStep{r.wheels, 0, (uint32_t)r.count};
        mark_filled(d);
        launch_relayout_chain(r.rt->stream, d->ptr, r.src->ptr, eb, c);
      } else {
        fill_pending(r.rt, r.dst);  // cells the views leave dead read as zero
        launch_relayout(r.rt->stream, r.dst->ptr, r.src->ptr, eb, 0, 0, r.count, r.wheels);
      }
    } else if (is_chain(r)) {
      for (int k = 0; k < r.pre.n; ++k)
        launch_map(r.rt->stream, r.dst->ptr, FO_F32, k == 0 ? r.src->ptr : r.dst->ptr, FO_F32, r.n, r.pre.op[k]);
    } else
      launch_map(r.rt->stream, r.dst->ptr, r.dst_t, r.src->ptr, r.src_t, r.n, r.op);
    const_cast<fo_buffer*>(r.dst)->widen_pending = false;
  }
}

// Narrow and broadcast records that have run serve nothing (only deferred ones are read through).
void drop_run_narrows() {
  std::vector<fo_buffer*> gone;
  {
    std::lock_guard<std::mutex> lock(g_widen_mu);
    gone = erase_records([](const WidenRecord& r) { return (is_narrow(r) || r.kind != 0) && !r.deferred; });
  }
  free_retired(gone);
}

// b is about to be written: a deferred cast into it (the write may be partial) and the deferred
// casts that read it run first, each after the casts its own source waits for; then b's records go.
void note_write(const fo_buffer* b) {
  if (!b) return;
  std::vector<const fo_buffer*> readers;
  {
    std::lock_guard<std::mutex> lock(g_widen_mu);
    for (auto& r : g_widen)
      if (r.src == b && r.deferred && r.dst != b) readers.push_back(r.dst);
  }
  materialize(b);
  for (const fo_buffer* d : readers) materialize(d);
  std::vector<fo_buffer*> gone;
  {
    std::lock_guard<std::mutex> lock(g_widen_mu);
    gone = erase_records([b](const WidenRecord& r) { return r.dst == b || r.src == b; });
  }
  free_retired(gone);
}

// b is about to be overwritten whole: the deferred casts that read it run first (each after the
// casts its own source waits for); a deferred op into it is dropped, since nothing can read its
// result any more.
void note_overwrite(const fo_buffer* b) {
  if (!b) return;
  std::vector<const fo_buffer*> readers;
  {
    std::lock_guard<std::mutex> lock(g_widen_mu);
    for (auto& r : g_widen)
      if (r.src == b && r.deferred && r.dst != b) readers.push_back(r.dst);
  }
  for (const fo_buffer* d : readers) materialize(d);
  std::vector<fo_buffer*> gone;
  {
    std::lock_guard<std::mutex> lock(g_widen_mu);
    gone = erase_records([b](const WidenRecord& r) { return r.dst == b || r.src == b; });
  }
  const_cast<fo_buffer*>(b)->widen_pending = false;
  free_retired(gone);
}

// b is being freed and no record reads it (retire_source keeps it otherwise): a cast into it is
// dropped.
void forget_buffer(const fo_buffer* b) {
  std::vector<fo_buffer*> gone;
  {
    std::lock_guard<std::mutex> lock(g_widen_mu);
    gone = erase_records([b](const WidenRecord& r) { return r.dst == b || r.src == b; });
  }
  free_retired(gone);
}

// b is being freed while a record reads it as its source: it is kept (retired), so the cast can stay
// deferred and a contraction can still read the narrow data; the block is freed when the last such
// record goes. Returns false (nothing kept) when no record reads b.
bool retire_source(fo_buffer* b) {
  std::lock_guard<std::mutex> lock(g_widen_mu);
  if (!std::any_of(g_widen.begin(), g_widen.end(), [b](const WidenRecord& r) { return r.src == b; })) return false;
  b->retired = true;
  if (b->pool) {
    std::lock_guard<std::mutex> plock(b->pool->mu);
    b->retired_in = b->pool->recording;
  }
  g_retired.push_back(b);
  return true;
}

// A record whose cast has run says dst = cast(src) only while neither buffer has been written
// since; eager writes drop it (note_write), but a graph launch writes buffers without telling the
// records. So before a recording starts (a recorded kernel must not read src in place of a dst that
// later eager writes may make differ from it) and before a graph launches (later eager calls must
// not take a replayed write of src or dst for the cast), every record that has run is dropped;
// retired sources that no record reads any more go with them, so that no recorded kernel reads a
// block the recording does not own.
void drop_run_records() {
  std::vector<fo_buffer*> gone;
  {
    std::lock_guard<std::mutex> lock(g_widen_mu);
    gone = erase_records([](const WidenRecord& r) { return !r.deferred; });
  }
  free_retired(gone);
}

// b is about to be read: its deferred cast, if any, runs first (a widen record stays for
// contractions).
void materialize(const fo_buffer* b) {
  if (!b->widen_pending) return;
  std::vector<WidenRecord> todo;
  {
    std::lock_guard<std::mutex> lock(g_widen_mu);
    for (auto& r : g_widen)
      if (r.dst == b && r.deferred) {
        todo.push_back(r);
        r.deferred = false;
      }
  }
  run_deferred(todo);
  drop_run_narrows();
}

// A runtime going away, or a recording starting or ending: every cast it deferred runs now, on its
// stream.
void materialize_runtime(fo_runtime* rt) {
  std::vector<WidenRecord> todo;
  {
    std::lock_guard<std::mutex> lock(g_widen_mu);
    for (auto& r : g_widen)
      if (r.rt == rt && r.deferred) {
        todo.push_back(r);
        r.deferred = false;
      }
  }
  run_deferred(todo);
  drop_run_narrows();
}

void record_widen(fo_runtime* rt, fo_buffer* dst, const fo_buffer* src, fo_dtype dst_t, fo_dtype src_t, uint64_t n,
                  const fo_op& op) {
  std::lock_guard<std::mutex> lock(g_widen_mu);
  g_widen.push_back({dst, src, src_t, n, dst_t, op, rt, true});
  dst->widen_pending = true;
}

// b holds a widen of at least n bf16 elements into f32, recorded on rt and not yet run.
bool deferred_bf16_widen(const fo_runtime* rt, const fo_buffer* b, uint64_t n, WidenRecord* out) {
  if (!b || !b->widen_pending) return false;
  std::lock_guard<std::mutex> lock(g_widen_mu);
  for (auto& r : g_widen)
    if (r.dst == b && r.deferred) {
      if (r.rt != rt || r.kind != 0 || r.src_t != FO_BF16 || r.dst_t != FO_F32 || r.op.code != FO_OP_CAST || r.n < n)
        return false;
      *out = r;
      return true;
    }
  return false;
}

// b holds a narrow of at least n f32 elements into bf16, recorded on rt and not yet run.
bool deferred_bf16_narrow(const fo_runtime* rt, const fo_buffer* b, uint64_t n, WidenRecord* out) {
  if (!b || !b->widen_pending) return false;
  std::lock_guard<std::mutex> lock(g_widen_mu);
  for (auto& r : g_widen)
    if (r.dst == b && r.deferred) {
      if (r.rt != rt || !is_narrow(r) || r.op.code != FO_OP_CAST || r.n < n) return false;
      *out = r;
      return true;
    }
  return false;
}

// b holds a broadcast of at least n elements, recorded on rt and not yet run.
bool deferred_bcast(const fo_runtime* rt, const fo_buffer* b, uint64_t n, WidenRecord* out) {
  if (!b || !b->widen_pending) return false;
  std::lock_guard<std::mutex> lock(g_widen_mu);
  for (auto& r : g_widen)
    if (r.dst == b && r.deferred) {
      if (r.rt != rt || !is_bcast(r) || r.n < n) return false;
      *out = r;
      return true;
    }
  return false;
}

// b holds a chain of f32 maps over at least n elements, recorded on rt and not yet run.
bool deferred_chain(const fo_runtime* rt, const fo_buffer* b, uint64_t n, WidenRecord* out) {
  if (!b || !b->widen_pending) return false;
  std::lock_guard<std::mutex> lock(g_widen_mu);
  for (auto& r : g_widen)
    if (r.dst == b && r.deferred) {
      if (r.rt != rt || !is_chain(r) || r.n < n) return false;
      *out = r;
      return true;
    }
  return false;
}

// b holds a recorded relayout, recorded on rt and not yet run.
bool deferred_xpose(const fo_runtime* rt, const fo_buffer* b, WidenRecord* out) {
  if (!b || !b->widen_pending) return false;
  std::lock_guard<std::mutex> lock(g_widen_mu);
  for (auto& r : g_widen)
    if (r.dst == b && r.deferred) {
      if (r.rt != rt || !is_xpose(r)) return false;
      *out = r;
      return true;
    }
  return false;
}

// How a zip, map or reduce reads an f32 input b of n elements (dst: the op's output, which the read
// must not alias): the buffer itself (code 4), the bf16 source of its deferred widen (2), or the f32
// source of that bf16's deferred narrow (kReadViaBf16); for a zip (bcast_ok) b may also be a
// deferred broadcast, read through its index map (div, mod) from its source, itself read as above;
// and (zip: chain_ok) the f32 data read, or narrowed, may be a deferred chain of f32 maps, applied
// on load (pre) to its source. `buf` is what the kernel reads and what the caller checks (which runs
// whatever is still deferred into it).
struct F32Read {
  const fo_buffer* buf;
  int code;
  uint32_t div = 1, mod = 0;
  PreOps pre{};
};
F32Read f32_read(const fo_runtime* rt, const fo_buffer* b, uint64_t n, const fo_buffer* dst, bool bcast_ok = false,
                 bool chain_ok = false) {
  WidenRecord br{}, ch{};
  if (bcast_ok && deferred_bcast(rt, b, n, &br) && br.src != dst) {
    F32Read s = f32_read(rt, br.src, br.mod, dst, false, chain_ok);
    s.div = br.div;
    s.mod = br.mod;
    return s;
  }
  if (chain_ok && deferred_chain(rt, b, n, &ch) && ch.src != dst) return {ch.src, 4, 1, 0, ch.pre};
  WidenRecord w{}, nr{};
  if (!deferred_bf16_widen(rt, b, n, &w) || w.src == dst) return {b, 4};
  if (deferred_bf16_narrow(rt, w.src, n, &nr) && nr.src != dst) {
    if (chain_ok && deferred_chain(rt, nr.src, n, &ch) && ch.src != dst) return {ch.src, kReadViaBf16, 1, 0, ch.pre};
    return {nr.src, kReadViaBf16};
  }
  return {w.src, 2};
}

bool find_widen(const fo_buffer* dst, WidenRecord* out) {
  std::lock_guard<std::mutex> lock(g_widen_mu);
  for (auto& r : g_widen)
    if (r.dst == dst && r.kind == 0 && !is_narrow(r)) {
      *out = r;
      return true;
    }
  return false;
}

template <typename F>
int32_t guard(F&& f) {
  try {
    f();
    g_last_error.clear();
    return FO_OK;
  } catch (const InvalidArg& e) {
    g_last_error = e.what();
    return FO_ERR_INVALID;
  } catch (const fm::Error& e) {
    g_last_error = e.what();
    return FO_ERR_INVALID;
  } catch (const HipError& e) {
    g_last_error = e.what();
    return FO_ERR_HIP;
  } catch (const OomError& e) {
    g_last_error = e.what();
    return FO_ERR_OOM;
  } catch (const Unsupported& e) {
    g_last_error = e.what();
    return FO_ERR_UNSUPPORTED;
  } catch (const std::exception& e) {
    g_last_error = e.what();
    return FO_ERR_INVALID;
  }
}

int64_t write_str(const std::string& s, char* out, uint64_t cap) {
  if (out && cap) {
    size_t n = std::min<size_t>(s.size(), cap - 1);
    std::memcpy(out, s.data(), n);
    out[n] = 0;
  }
  return (int64_t)s.size();
}

// Mapping work memoised by the strings that determine it: an engine issues the same few layouts
// over and over, so each is parsed and resolved once per process (a failing one is not kept and
// fails again on the next call). The table is cleared when it reaches its cap.
template <typename V>
class Memo {
  std::mutex mu_;
  std::unordered_map<std::string, V> m_;
  static constexpr size_t kCap = 4096;

 public:
  template <typename F>
  V get(const std::string& key, F&& make) {
    {
      std::lock_guard<std::mutex> lock(mu_);
      auto it = m_.find(key);
      if (it != m_.end()) return it->second;
    }
    V v = make();
    std::lock_guard<std::mutex> lock(mu_);
    if (m_.size() >= kCap) m_.clear();
    m_.emplace(key, v);
    return v;
  }
};

// The key of several strings (NUL-free C strings, NULL read as empty).
std::string memo_key(std::initializer_list<const char*> parts) {
  std::string k;
  for (const char* p : parts) {
    if (p) k += p;
    k += '\x01';
  }
  return k;
}

fm::Factors flat(const char* json_text, const char* what) {
  require(json_text && *json_text, std::string(what) + ": mapping is required");
  static Memo<fm::Factors> memo;
  return memo.get(json_text, [&] { return fm::flatten(fm::parse_json(json_text)); });
}

// The runtime of the entry point running on this thread (set by check_rt, which every entry point
// that takes buffers calls first): the stream a deferred zero fill goes on.
thread_local fo_runtime* t_rt = nullptr;
void check_rt(fo_runtime* rt) {
  require(rt != nullptr, "runtime is NULL");
  t_rt = rt;
}
// The buffer's zero fill has run or is no longer owed.
void mark_filled(fo_buffer* b) {
  b->zero_pending = false;
  if (b->pool) {
    std::lock_guard<std::mutex> lock(b->pool->mu);
    b->pool->unfilled.erase(b);
  }
}
void fill_pending(fo_runtime* rt, const fo_buffer* b) {
  if (!b->zero_pending) return;
  fo_buffer* m = const_cast<fo_buffer*>(b);
  FO_HIP(hipSetDevice(rt->device));
  launch_zero(rt->stream, m->ptr, (m->capacity + 15) & ~15ull);
  mark_filled(m);
}
void check_ptr(const fo_buffer* b, const char* what) {
  require(b != nullptr && b->ptr != nullptr, std::string(what) + " buffer is NULL");
}
// A buffer whose zero fill, if deferred, must run now (a deferred cast into it may stay deferred).
void check_filled(const fo_buffer* b, const char* what) {
  check_ptr(b, what);
  if (b->zero_pending) {
    require(t_rt != nullptr, "buffer used before any runtime call on this thread");
    fill_pending(t_rt, b);
  }
}
// A buffer an op reads, or writes in part: its deferred zero fill and any deferred cast into it go
// first.
void check_buf(const fo_buffer* b, const char* what) {
  check_filled(b, what);
  materialize(b);
}
// An op's output, just before its launch: `written` bytes from the start are overwritten; when
// they cover the buffer the deferred zero fill is dropped, otherwise it goes first.
void claim_out(fo_runtime* rt, fo_buffer* b, uint64_t written) {
  if (!b->zero_pending) return;
  if (written >= b->bytes)
    mark_filled(b);
  else
    fill_pending(rt, b);
}

// The recording open on rt's pool, if any (fo_graph_begin .. fo_graph_end).
fo_graph_mem* recording(const fo_runtime* rt) { return rt->pool ? rt->pool->recording.get() : nullptr; }
// Calls that wait for the device cannot be recorded into a graph.
void not_recording(const fo_runtime* rt, const char* what) {
  require(recording(rt) == nullptr,
          std::string(what) + " waits for the device: not allowed while a graph is being recorded");
}

// Size classes: 512-byte multiples below 1 MiB, 2 MiB multiples above. A free block serves a
// request of its class, or a large request up to a quarter smaller than the block.
uint64_t size_class(uint64_t need) {
  return need < (1ull << 20) ? (need + 511) & ~511ull : (need + (2ull << 20) - 1) & ~((2ull << 20) - 1);
}
bool fits(uint64_t block, uint64_t cls) { return block == cls || (cls >= (1ull << 20) && block - block / 4 <= cls); }

// A device block of at least `need` bytes, as (address, capacity): while recording, first from the
// blocks freed in the recording; then from the runtime's cache; else newly allocated. A block
// taken while recording joins the recording's memory.
std::pair<void*, uint64_t> take_block(fo_runtime* rt, uint64_t need) {
  const uint64_t cls = size_class(need ? need : 1);
  fo_graph_mem* rec = recording(rt);
  if (rec) {
    auto it = rec->reuse.lower_bound(cls);
    if (it != rec->reuse.end() && fits(it->first, cls)) {
      std::pair<void*, uint64_t> r{it->second, it->first};
      rec->reuse.erase(it);
      return r;  // already one of the recording's blocks
    }
  }
  void* ptr = nullptr;
  uint64_t cap = 0;
  {
    std::lock_guard<std::mutex> lock(rt->pool->mu);
    auto it = rt->pool->cached.lower_bound(cls);
    if (it != rt->pool->cached.end() && fits(it->first, cls)) {
      ptr = it->second;
      cap = it->first;
      rt->pool->cached_bytes -= it->first;
      rt->pool->cached.erase(it);
    }
  }
  if (!ptr) {
    hipError_t e = hipMalloc(&ptr, cls);
    if (e != hipSuccess && !rec) {
      // Release the cache (after the stream drains) and try once more.
      (void)hipGetLastError();
      FO_HIP(hipStreamSynchronize(rt->stream));
      std::lock_guard<std::mutex> lock(rt->pool->mu);
      for (auto& kv : rt->pool->cached) (void)hipFree(kv.second);
      rt->pool->cached.clear();
      rt->pool->cached_bytes = 0;
      e = hipMalloc(&ptr, cls);
    }
    if (e != hipSuccess) {
      (void)hipGetLastError();
      throw OomError("hipMalloc(" + std::to_string(cls) + ") failed: " + hipGetErrorString(e));
    }
    cap = cls;
  }
  if (rec) rec->blocks.emplace_back(cap, ptr);
  return {ptr, cap};
}

void set_device(fo_runtime* rt) { FO_HIP(hipSetDevice(rt->device)); }


// Hands the recorded spans to the sink (the stream has drained), then releases their events.
void flush_trace(fo_runtime* rt) {
  if (rt->spans.empty()) return;
  std::vector<fo_runtime::Span> spans;
  spans.swap(rt->spans);
  for (auto& sp : spans) {
    float b = 0.f, e = 0.f;
    if (rt->trace_sink && rt->trace_base && hipEventElapsedTime(&b, rt->trace_base, sp.begin) == hipSuccess &&
        hipEventElapsedTime(&e, rt->trace_base, sp.end) == hipSuccess)
      rt->trace_sink(rt->trace_ctx, sp.name, std::strlen(sp.name), (uint64_t)((double)b * 1e6),
                     (uint64_t)((double)e * 1e6));
    (void)hipEventDestroy(sp.begin);
    (void)hipEventDestroy(sp.end);
  }
  if (rt->trace_done) rt->trace_done(rt->trace_ctx);
}

// The live-digit sub-odometer of a wheel list (digits >= live are padding and never folded).
std::vector<fm::Wheel> live_only(const std::vector<fm::Wheel>& ws) {
  std::vector<fm::Wheel> out;
  for (auto w : ws) {
    if (w.live <= 1) continue;
    w.size = w.live;
    out.push_back(w);
  }
  return out;
}

// Adjacent fully live wheels that are contiguous in every memory (inner stride x inner size = outer
// stride) as one wheel: the same positions in the same order, fewer digits to decode. A residue
// split by the out axes of a pre-reduce mapping (H / 32, then H % 32 past a lane axis) comes back
// whole, and the kernels' unit-stride forms apply to it.
std::vector<fm::Wheel> merge_contiguous(const std::vector<fm::Wheel>& ws) {
  std::vector<fm::Wheel> out;
  for (const auto& w : ws) {
    if (!out.empty()) {
      fm::Wheel& in = out.back();
      bool ok = in.live == in.size && w.live == w.size && in.stride.size() == w.stride.size();
      for (size_t k = 0; ok && k < w.stride.size(); ++k) ok = in.stride[k] * in.size == w.stride[k];
      if (ok) {
        in.size *= w.size;
        in.live = in.size;
        continue;
      }
    }
    out.push_back(w);
  }
  return out;
}

std::vector<fm::Wheel> part(const fm::Joint& j, int p) {
  std::vector<fm::Wheel> out;
  for (auto& w : j.wheels)
    if (w.part == p) out.push_back(w);
  return out;
}

// Largest offset a walk over the live digits can reach in memory k (strides are >= 0).
int64_t max_live_offset(const std::vector<fm::Wheel>& ws, int k) {
  int64_t m = 0;
  for (auto& w : ws)
    if (w.live > 0) m += (w.live - 1) * w.stride[k];
  return m;
}

// The runtime's device scratch, at least `bytes` long (grown after the stream drains).
void* runtime_scratch(fo_runtime* rt, uint64_t bytes) {
  if (fo_graph_mem* rec = recording(rt)) {
    // The recording's own scratch: the eager one may be regrown (freed) while the graph lives.
    if (rec->scratch_bytes < bytes) {
      auto blk = take_block(rt, bytes);
      rec->scratch = blk.first;
      rec->scratch_bytes = blk.second;
    }
    return rec->scratch;
  }
  if (rt->scratch_bytes < bytes) {
    FO_HIP(hipStreamSynchronize(rt->stream));
    if (rt->scratch) FO_HIP(hipFree(rt->scratch));
    rt->scratch = nullptr;
    rt->scratch_bytes = 0;
    FO_HIP(hipMalloc(&rt->scratch, bytes));
    rt->scratch_bytes = bytes;
  }
  return rt->scratch;
}

// Waits for a graph's launches, then destroys it; its memory goes when its last buffer does.
void destroy_graph(fo_graph* g) {
  if (g->rt) {
    (void)hipSetDevice(g->rt->device);
    (void)hipStreamSynchronize(g->rt->stream);
    g->rt->graphs.erase(g);
  }
  if (g->exec) (void)hipGraphExecDestroy(g->exec);
  if (g->graph) (void)hipGraphDestroy(g->graph);
  delete g;
}

// The runtime's device-visible error word (pinned host memory, written by kernels only when an
// op's data is invalid). Returns its device address.
int32_t* error_word(fo_runtime* rt) {
  if (!rt->err_host) {
    void* h = nullptr;
    FO_HIP(hipHostMalloc(&h, sizeof(int32_t), hipHostMallocMapped));
    rt->err_host = (int32_t*)h;
    *rt->err_host = 0;
    void* d = nullptr;
    FO_HIP(hipHostGetDevicePointer(&d, h, 0));
    rt->err_dev = (int32_t*)d;
  }
  return rt->err_dev;
}
// Index errors of gather / scatter are found on the device. The op itself returns as soon as it is
// enqueued, like every other op; the next call that waits for the stream (fo_runtime_synchronize,
// fo_read) reports the error and clears the word. Call after the stream has drained.
void raise_device_errors(fo_runtime* rt) {
  if (!rt->err_ops) return;
  const uint32_t ops = rt->err_ops;
  rt->err_ops = 0;
  if (__atomic_load_n(rt->err_host, __ATOMIC_ACQUIRE) == 0) return;
  __atomic_store_n(rt->err_host, 0, __ATOMIC_RELEASE);
  // Each op that may have set the word names its own failure (the word does not say which op set it).
  std::string msg;
  if (ops & 3u)
    msg = std::string((ops & 3u) == 1u ? "gather" : (ops & 3u) == 2u ? "scatter" : "gather or scatter") +
          ": an index is negative or past the indexed axis (the valid indices were applied)";
  if (ops & 4u)
    msg += std::string(msg.empty() ? "" : "; or ") +
           "zip3_slots: a tag byte above 15 is not an execution id (that cell passed through)";
  throw InvalidArg(msg + " -- in an op issued since the last synchronization");
}

// Shared set-up of scatter / gather: the stream wheels of one side. A pad of the stream (an interior
// pad of the payload, such as the 1 # 32 of a [N, 1 # 32, D] slice placement) that no memory cell
// backs is a wheel of stride 0: SequencerConfig::iter (furiosa-mapping-types/src/lib.rs:866-905)
// walks its positions as repeats of the live one, so they repeat its reads and writes. A pad that
// memory backs would read or write pad cells: refused.
std::vector<fm::Wheel> stream_wheels(const fm::Factors& memory, const fm::Factors& outer, const fm::Factors& inner,
                                     const char* what) {
  fm::Joint j = fm::sequence({memory}, {outer, inner}, fm::Mode::Read);
  for (auto& w : j.wheels)
    require(w.live == w.size || w.stride[0] == 0,
            std::string(what) + ": a stream pad that memory backs is not supported");
  return j.wheels;
}

// Number of innermost wheels from the inner stream part (part 1): the outer part's follow them.
int inner_part_wheels(const std::vector<fm::Wheel>& ws) {
  int n = 0;
  while (n < (int)ws.size() && ws[n].part == 1) ++n;
  return n;
}

int64_t product(const std::vector<fm::Wheel>& ws) {
  int64_t p = 1;
  for (auto& w : ws) p *= w.size;
  return p;
}

// ---- safetensors -----------------------------------------------------------------------------
// safetensors host loading at the boundary: HostTensor::from_safetensors (furiosa-opt-std/src/
// tensor/memory.rs:190-223) for a file on disk, so weights reach HBM without a host-side copy of
// the whole file in another format.
//
// File layout (the safetensors format): an 8-byte little-endian header length N, N bytes of JSON
// mapping each tensor name to {"dtype", "shape", "data_offsets": [begin, end]} (offsets relative to
// the byte after the header; an optional "__metadata__" entry), then the data. The reference
// checks the view's shape against the pair-flattened sizes of the element mapping and its byte
// length against the mapping's size; the bytes are then the packed device image as they are.

struct TensorInfo {
  std::string dtype;
  std::vector<int64_t> shape;
  uint64_t begin = 0, end = 0;  // absolute file offsets of the data
};

struct File {
  FILE* f = nullptr;
  explicit File(const char* path) : f(std::fopen(path, "rb")) {}
  ~File() {
    if (f) std::fclose(f);
  }
};

TensorInfo find_tensor(File& file, const char* path, const char* name) {
  require(file.f != nullptr, std::string("safetensors: cannot open '") + path + "'");
  unsigned char len8[8];
  require(std::fread(len8, 1, 8, file.f) == 8, "safetensors: file shorter than its header length");
  uint64_t n = 0;
  for (int i = 7; i >= 0; --i) n = (n << 8) | len8[i];
  require(n > 0 && n < (1ull << 30), "safetensors: implausible header length");
  std::string header(n, '\0');
  require(std::fread(&header[0], 1, n, file.f) == n, "safetensors: truncated header");
  std::fseek(file.f, 0, SEEK_END);
  const uint64_t file_size = (uint64_t)std::ftell(file.f);
  fo::json::Value h = fo::json::parse(header);
  require(h.kind == fo::json::Value::Object, "safetensors: the header is not a JSON object");
  const fo::json::Value* t = h.get(name);
  require(t != nullptr && std::string(name) != "__metadata__", std::string("safetensors: no tensor '") + name + "'");
  TensorInfo info;
  info.dtype = t->at("dtype").as_str();
  for (auto& d : t->at("shape").arr) info.shape.push_back(d.as_int());
  const fo::json::Value& off = t->at("data_offsets");
  require(off.kind == fo::json::Value::Array && off.arr.size() == 2, "safetensors: data_offsets is not a pair");
  const int64_t b = off.arr[0].as_int(), e = off.arr[1].as_int();
  require(b >= 0 && e >= b, "safetensors: bad data_offsets");
  info.begin = 8 + n + (uint64_t)b;
  info.end = 8 + n + (uint64_t)e;
  require(info.end <= file_size, "safetensors: data_offsets past the end of the file");
  return info;
}

// flat_shape (memory.rs:204-212): a Pair contributes its two sides, anything else its size.
void flat_shape(const fm::NodeP& m, std::vector<int64_t>& out) {
  if (m->kind == fm::Node::Pair) {
    flat_shape(m->a, out);
    flat_shape(m->b, out);
  } else {
    out.push_back(fm::size(m));
  }
}

int32_t dtype_code(const std::string& s) {
  if (s == "I8") return FO_I8;
  if (s == "U8") return FO_U8;
  if (s == "I16") return FO_I16;
  if (s == "I32") return FO_I32;
  if (s == "BF16") return FO_BF16;
  if (s == "F32") return FO_F32;
  if (s == "F8_E4M3") return FO_F8E4M3;
  if (s == "F8_E5M2") return FO_F8E5M2;
  return -1;
}

}  // namespace

extern "C" {

const char* fo_last_error(void) { return g_last_error.c_str(); }

int32_t fo_runtime_init(int32_t device_index, fo_runtime** out) {
  return guard([&] {
    require(out != nullptr, "out is NULL");
    *out = nullptr;
    int n = 0;
    FO_HIP(hipGetDeviceCount(&n));
    require(device_index >= 0 && device_index < n,
            "device index " + std::to_string(device_index) + " out of range (" + std::to_string(n) + " devices)");
    auto* rt = new fo_runtime();
    rt->device = device_index;
    rt->pool = std::make_shared<fo_pool>();
    rt->pool->device = device_index;
    try {
      FO_HIP(hipSetDevice(device_index));
      static_scratch_init(device_index);
      FO_HIP(hipStreamCreateWithFlags(&rt->stream, hipStreamNonBlocking));
      for (auto& e : rt->events) FO_HIP(hipEventCreate(&e));
      hipDeviceProp_t prop;
      FO_HIP(hipGetDeviceProperties(&prop, device_index));
      rt->cus = prop.multiProcessorCount;
      rt->arch = prop.gcnArchName;
      FO_HIP(hipMalloc((void**)&rt->gemm_ws.parts, fo::GemmWorkspace::kBytes));
      FO_HIP(hipMalloc((void**)&rt->gemm_ws.arrived, fo::GemmWorkspace::kTiles * sizeof(uint32_t)));
      launch_zero(rt->stream, rt->gemm_ws.arrived, fo::GemmWorkspace::kTiles * sizeof(uint32_t));
      const char* eager = getenv("FO_EAGER");
      rt->eager = eager && *eager && std::strcmp(eager, "0") != 0;
    } catch (...) {
      fo_runtime_free(rt);
      throw;
    }
    *out = rt;
  });
}

void fo_runtime_free(fo_runtime* rt) {
  if (!rt) return;
  (void)hipSetDevice(rt->device);
  if (rt->pool && rt->pool->recording) {  // an open recording is discarded
    hipGraph_t g = nullptr;
    (void)hipStreamEndCapture(rt->stream, &g);
    if (g) (void)hipGraphDestroy(g);
    (void)hipGetLastError();
    std::lock_guard<std::mutex> lock(rt->pool->mu);
    rt->pool->recording.reset();
  }
  for (fo_graph* g : rt->graveyard) destroy_graph(g);
  rt->graveyard.clear();
  // Graphs still held by the caller lose their executables; fo_graph_free then only releases them.
  for (fo_graph* g : rt->graphs) {
    (void)hipStreamSynchronize(rt->stream);
    if (g->exec) (void)hipGraphExecDestroy(g->exec);
    if (g->graph) (void)hipGraphDestroy(g->graph);
    g->exec = nullptr;
    g->graph = nullptr;
    g->rt = nullptr;
  }
  rt->graphs.clear();
  try {
    materialize_runtime(rt);
  } catch (const std::exception&) {
  }
  if (rt->stream) (void)hipStreamSynchronize(rt->stream);
  for (auto& e : rt->events)
    if (e) (void)hipEventDestroy(e);
  for (auto& sp : rt->spans) {
    (void)hipEventDestroy(sp.begin);
    (void)hipEventDestroy(sp.end);
  }
  if (rt->trace_base) (void)hipEventDestroy(rt->trace_base);
  if (rt->scratch) (void)hipFree(rt->scratch);
  if (rt->gemm_ws.parts) (void)hipFree(rt->gemm_ws.parts);
  if (rt->gemm_ws.arrived) (void)hipFree(rt->gemm_ws.arrived);
  if (rt->pool) {
    std::lock_guard<std::mutex> lock(rt->pool->mu);
    for (auto& kv : rt->pool->cached) (void)hipFree(kv.second);
    rt->pool->cached.clear();
    rt->pool->cached_bytes = 0;
    rt->pool->orphaned = true;
  }
  if (rt->scatter_win) (void)hipFree(rt->scatter_win);
  if (rt->err_host) (void)hipHostFree(rt->err_host);
  if (rt->stream) (void)hipStreamDestroy(rt->stream);
  delete rt;
}

int32_t fo_runtime_synchronize(fo_runtime* rt) {
  return guard([&] {
    check_rt(rt);
    not_recording(rt, "fo_runtime_synchronize");
    FO_HIP(hipStreamSynchronize(rt->stream));
    flush_trace(rt);
    raise_device_errors(rt);
  });
}

int32_t fo_runtime_set_trace(fo_runtime* rt, fo_trace_sink sink, fo_trace_done done, void* ctx) {
  return guard([&] {
    check_rt(rt);
    not_recording(rt, "fo_runtime_set_trace");
    set_device(rt);
    FO_HIP(hipStreamSynchronize(rt->stream));
    flush_trace(rt);  // spans of the previous sink go to it
    if (rt->trace_base) {
      (void)hipEventDestroy(rt->trace_base);
      rt->trace_base = nullptr;
    }
    rt->trace_sink = sink;
    rt->trace_done = done;
    rt->trace_ctx = ctx;
    if (sink) {
      FO_HIP(hipEventCreate(&rt->trace_base));
      FO_HIP(hipEventRecord(rt->trace_base, rt->stream));
    }
  });
}

int32_t fo_runtime_device_info(fo_runtime* rt, int32_t* compute_units, char* arch, uint64_t arch_cap) {
  return guard([&] {
    check_rt(rt);
    if (compute_units) *compute_units = rt->cus;
    write_str(rt->arch, arch, arch_cap);
  });
}

int32_t fo_buffer_alloc(fo_runtime* rt, uint64_t bytes, fo_buffer** out) {
  return guard([&] {
    check_rt(rt);
    require(out != nullptr, "out is NULL");
    *out = nullptr;
    set_device(rt);
    auto b = std::make_unique<fo_buffer>();
    b->bytes = bytes;
    b->device = rt->device;
    b->pool = rt->pool;
    auto blk = take_block(rt, bytes);
    b->ptr = blk.first;
    b->capacity = blk.second;
    b->graph_mem = rt->pool->recording;  // null unless a graph is being recorded
    // Zero-filled (Backend::zeroed), the fill deferred to the first use (check_buf / claim_out). It
    // then runs on that op's runtime stream, after every earlier op of the runtime, including a
    // reuse's previous owner's last reads.
    b->zero_pending = true;
    {
      std::lock_guard<std::mutex> lock(rt->pool->mu);
      rt->pool->unfilled.insert(b.get());
    }
    if (rt->eager) fill_pending(rt, b.get());
    *out = b.release();
  });
}

void fo_buffer_free(fo_buffer* buf) {
  if (!buf) return;
  if (retire_source(buf)) return;
  try {
    forget_buffer(buf);
  } catch (const std::exception&) {  // a failed launch leaves the error for the next call to report
  }
  std::shared_ptr<fo_graph_mem> rec;
  if (buf->pool) {
    std::lock_guard<std::mutex> lock(buf->pool->mu);
    rec = buf->pool->recording;
  }
  free_block(buf, rec);
}

int32_t fo_buffer_clone(fo_runtime* rt, const fo_buffer* src, fo_buffer** out) {
  return guard([&] {
    check_rt(rt);
    check_buf(src, "src");
    require(out != nullptr, "out is NULL");
    fo_buffer* b = nullptr;
    int32_t st = fo_buffer_alloc(rt, src->bytes, &b);
    if (st != FO_OK) throw OomError(g_last_error);
    mark_filled(b);  // every byte is copied
    FO_HIP(hipMemcpyAsync(b->ptr, src->ptr, src->bytes, hipMemcpyDeviceToDevice, rt->stream));
    *out = b;
  });
}

uint64_t fo_buffer_bytes(const fo_buffer* buf) { return buf ? buf->bytes : 0; }

int32_t fo_buffer_flush(fo_runtime* rt, const fo_buffer* buf) {
  return guard([&] {
    check_rt(rt);
    check_buf(buf, "buf");
  });
}

int32_t fo_write(fo_runtime* rt, const void* host, uint64_t bytes, fo_buffer* dst) {
  return guard([&] {
    check_rt(rt);
    not_recording(rt, "fo_write");
    check_ptr(dst, "dst");
    note_write(dst);
    require(host != nullptr || bytes == 0, "host pointer is NULL");
    require(bytes <= dst->bytes, "write of " + std::to_string(bytes) + " bytes exceeds the buffer");
    set_device(rt);
    claim_out(rt, dst, bytes);
    TraceScope trace_span(rt, "write");
    FO_HIP(hipMemcpyAsync(dst->ptr, host, bytes, hipMemcpyHostToDevice, rt->stream));
    FO_HIP(hipStreamSynchronize(rt->stream));
  });
}

int32_t fo_read(fo_runtime* rt, const fo_buffer* src, void* host, uint64_t bytes) {
  return guard([&] {
    check_rt(rt);
    not_recording(rt, "fo_read");
    check_buf(src, "src");
    require(host != nullptr || bytes == 0, "host pointer is NULL");
    require(bytes <= src->bytes, "read of " + std::to_string(bytes) + " bytes exceeds the buffer");
    set_device(rt);
    TraceScope trace_span(rt, "read");
    FO_HIP(hipMemcpyAsync(host, src->ptr, bytes, hipMemcpyDeviceToHost, rt->stream));
    FO_HIP(hipStreamSynchronize(rt->stream));
    raise_device_errors(rt);
  });
}

int32_t fo_event_record(fo_runtime* rt, int32_t slot) {
  return guard([&] {
    check_rt(rt);
    not_recording(rt, "fo_event_record");
    require(slot >= 0 && slot < 16, "event slot out of range");
    FO_HIP(hipEventRecord(rt->events[slot], rt->stream));
  });
}

int32_t fo_event_elapsed_ms(fo_runtime* rt, int32_t start, int32_t end, float* ms) {
  return guard([&] {
    check_rt(rt);
    not_recording(rt, "fo_event_elapsed_ms");
    require(start >= 0 && start < 16 && end >= 0 && end < 16, "event slot out of range");
    require(ms != nullptr, "ms is NULL");
    FO_HIP(hipEventSynchronize(rt->events[end]));
    FO_HIP(hipEventElapsedTime(ms, rt->events[start], rt->events[end]));
  });
}

// ---- recorded op streams -----------------------------------------------------------------------

int32_t fo_graph_begin(fo_runtime* rt) {
  return guard([&] {
    check_rt(rt);
    require(recording(rt) == nullptr, "a graph is already being recorded on this runtime");
    require(rt->trace_sink == nullptr, "trace spans are not recorded into graphs: clear the trace sink first");
    set_device(rt);
    // Everything owed to buffers that exist now runs eagerly, outside the graph: a launch must not
    // zero a cache that earlier launches filled, or redo a cast whose source has changed since.
    materialize_runtime(rt);
    drop_run_records();
    std::vector<fo_buffer*> unfilled;
    {
      std::lock_guard<std::mutex> lock(rt->pool->mu);
      unfilled.assign(rt->pool->unfilled.begin(), rt->pool->unfilled.end());
    }
    for (fo_buffer* b : unfilled) fill_pending(rt, b);
    (void)error_word(rt);
    auto mem = std::make_shared<fo_graph_mem>();
    mem->pool = rt->pool;
    FO_HIP(hipStreamBeginCapture(rt->stream, hipStreamCaptureModeRelaxed));
    rt->err_ops_saved = rt->err_ops;
    rt->err_ops = 0;
    std::lock_guard<std::mutex> lock(rt->pool->mu);
    rt->pool->recording = std::move(mem);
  });
}

int32_t fo_graph_end(fo_runtime* rt, fo_graph** out) {
  return guard([&] {
    check_rt(rt);
    require(out != nullptr, "out is NULL");
    *out = nullptr;
    require(recording(rt) != nullptr, "no graph is being recorded on this runtime");
    set_device(rt);
    // Casts deferred while recording whose outputs are still alive belong to the graph.
    std::string failure;
    try {
      materialize_runtime(rt);
    } catch (const std::exception& e) {
      failure = e.what();
    }
    hipGraph_t graph = nullptr;
    const hipError_t e = hipStreamEndCapture(rt->stream, &graph);
    std::shared_ptr<fo_graph_mem> mem;
    {
      std::lock_guard<std::mutex> lock(rt->pool->mu);
      mem = std::move(rt->pool->recording);
      rt->pool->recording.reset();
    }
    const uint32_t err_ops = rt->err_ops;
    rt->err_ops = rt->err_ops_saved;
    for (fo_graph* g : rt->graveyard) destroy_graph(g);
    rt->graveyard.clear();
    if (e != hipSuccess || graph == nullptr || !failure.empty()) {
      if (graph) (void)hipGraphDestroy(graph);
      (void)hipGetLastError();
      throw HipError(!failure.empty() ? failure
                                      : std::string("recording failed: hipStreamEndCapture: ") + hipGetErrorString(e));
    }
    hipGraphExec_t exec = nullptr;
    const hipError_t ie = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    if (ie != hipSuccess) {
      (void)hipGraphDestroy(graph);
      throw HipError(std::string("hipGraphInstantiate failed: ") + hipGetErrorString(ie));
    }
    auto* g = new fo_graph();
    g->rt = rt;
    g->graph = graph;
    g->exec = exec;
    g->mem = std::move(mem);
    g->err_ops = err_ops;
    rt->graphs.insert(g);
    *out = g;
  });
}

int32_t fo_graph_launch(fo_runtime* rt, fo_graph* graph) {
  return guard([&] {
    check_rt(rt);
    require(graph != nullptr, "graph is NULL");
    require(graph->rt == rt && graph->exec != nullptr, "the graph was not recorded on this runtime");
    require(recording(rt) == nullptr, "a graph cannot be launched while one is being recorded");
    set_device(rt);
    materialize_runtime(rt);  // casts deferred since, which the graph may read
    drop_run_records();
    TraceScope trace_span(rt, "graph");
    FO_HIP(hipGraphLaunch(graph->exec, rt->stream));
    rt->err_ops |= graph->err_ops;
  });
}

void fo_graph_free(fo_graph* graph) {
  if (!graph) return;
  if (graph->rt && recording(graph->rt)) {  // no waiting on a stream that is recording
    graph->rt->graveyard.push_back(graph);
    return;
  }
  destroy_graph(graph);
}

// ---- mapping utilities -------------------------------------------------------------------------

int64_t fo_mapping_parse(const char* text, const char* axes_json, char* out, uint64_t cap) {
  int64_t len = 0;
  int32_t st = guard([&] {
    require(text != nullptr, "text is NULL");
    std::map<std::string, int64_t> sizes;
    if (axes_json && *axes_json) {
      json::Value v = json::parse(axes_json);
      require(v.kind == json::Value::Object, "axes must be a JSON object");
      for (auto& kv : v.obj) sizes[kv.first] = kv.second.as_int();
    }
    len = write_str(fm::to_json(fm::parse_text(text, sizes)), out, cap);
  });
  return st == FO_OK ? len : st;
}

int32_t fo_mapping_sequence(const char* memory, const char* stream, int32_t mode, int64_t* sizes, int64_t* lives,
                            int64_t* strides, int32_t cap) {
  int32_t n = 0;
  int32_t st = guard([&] {
    require(mode >= 0 && mode <= 2, "mode must be 0 (Read), 1 (Write) or 2 (Carve)");
    fm::Joint j = fm::sequence({flat(memory, "memory")}, {flat(stream, "stream")}, (fm::Mode)mode);
    n = (int32_t)j.wheels.size();
    for (int32_t i = 0; i < n && i < cap; ++i) {
      if (sizes) sizes[i] = j.wheels[i].size;
      if (lives) lives[i] = j.wheels[i].live;
      if (strides) strides[i] = j.wheels[i].stride[0];
    }
  });
  return st == FO_OK ? n : st;
}

int64_t fo_mapping_carve(const char* self_map, const char* piece, char* out, uint64_t cap) {
  int64_t len = 0;
  int32_t st = guard([&] {
    fm::Factors c = fm::carve(flat(self_map, "self"), flat(piece, "piece"));
    len = write_str(fm::to_json(fm::unflatten(c)), out, cap);
  });
  return st == FO_OK ? len : st;
}

int64_t fo_mapping_window_base(const char* base_map, const char* offset) {
  int64_t base = 0;
  int32_t st = guard([&] {
    base = fm::window_base(flat(base_map, "base"), fm::parse_offset_json(offset ? offset : ""));
  });
  return st == FO_OK ? base : st;
}

// ---- elementwise ---------------------------------------------------------------------------------

int32_t fo_map(fo_runtime* rt, fo_buffer* dst, fo_dtype dst_t, const fo_buffer* src, fo_dtype src_t, uint64_t n,
               const fo_op* op) {
  return guard([&] {
    check_rt(rt);
    check_ptr(dst, "dst");
    note_write(dst);
    require(op != nullptr, "op is NULL");
    check_ptr(src, "src");
    require(span_bytes(dst_t, n) <= dst->bytes && span_bytes(src_t, n) <= src->bytes, "map: n exceeds a buffer");
    // An f32 input that stands for a deferred cast (a widen of bf16 data, maybe of a deferred
    // narrow) is read from the data it stands for, and the casts need not run.
    const F32Read rs = src_t == FO_F32 && (dst_t == FO_F32 || dst_t == FO_BF16) ? f32_read(rt, src, n, dst)
                                                                               : F32Read{src, 4};
    // An exact widening cast (the engine's contract_outer widen), or a narrowing cast of f32 data to
    // bf16, is recorded and deferred until something reads its output other than through it. Its
    // source gets its zero fill now; a deferred cast into the source stays deferred (running this
    // one runs that one first).
    const bool widen = !rt->eager && op->code == FO_OP_CAST && dst != src &&
                       ((dst_t == FO_F32 && (src_t == FO_BF16 || src_t == FO_F8E4M3 || src_t == FO_F8E5M2)) ||
                        (dst_t == FO_I32 && src_t == FO_I8) || (dst_t == FO_BF16 && src_t == FO_F32 && rs.code == 4));
    // An f32 -> f32 map of f32 data with nothing deferred into it, or of a deferred chain of fewer
    // than three such maps, is recorded as a chain (extended by this op) that a zip applies on load.
    WidenRecord ch{};
    bool chain = false;
    if (!rt->eager && src_t == FO_F32 && dst_t == FO_F32 && dst != src && op->code != FO_OP_CAST && op->code != FO_OP_CAST_RELU &&
        op->code != FO_OP_TABLE_LOOKUP && op->code != FO_OP_ZERO_POINT_SUB && op->code != FO_OP_FXP_TO_FP &&
        op->code != FO_OP_FP_TO_FXP) {
      if (!src->widen_pending) {
        ch.src = src;
        chain = true;
      } else if (deferred_chain(rt, src, n, &ch) && ch.pre.n < 3 && ch.src != dst) {
        chain = true;
      }
    }
    if (chain) {
      check_filled(ch.src, "src");
      if (n == 0) return;
      set_device(rt);
      claim_out(rt, dst, span_bytes(dst_t, n));
      std::lock_guard<std::mutex> lock(g_widen_mu);
      WidenRecord r{dst, ch.src, FO_F32, n, FO_F32, *op, rt, true};
      r.kind = 2;
      r.pre = ch.pre;
      r.pre.op[r.pre.n++] = *op;
      g_widen.push_back(r);
      dst->widen_pending = true;
      return;
    }
    if (widen)
      check_filled(src, "src");
    else
      check_buf(rs.buf, "src");
    if (n == 0) return;
    set_device(rt);
    claim_out(rt, dst, span_bytes(dst_t, n));
    if (widen) {
      record_widen(rt, dst, src, dst_t, src_t, n, *op);
      return;
    }
    TraceScope trace_span(rt, "map");
    if (rs.code != 4)
      launch_map_widened(rt->stream, dst->ptr, dst_t, rs.buf->ptr, rs.code, n, *op);
    else
      launch_map(rt->stream, dst->ptr, dst_t, src->ptr, src_t, n, *op);
  });
}

int32_t fo_zip_with(fo_runtime* rt, fo_buffer* dst, fo_dtype dst_t, const fo_buffer* a, const fo_buffer* b,
                    fo_dtype in_t, uint64_t n, const fo_op* op) {
  return guard([&] {
    check_rt(rt);
    check_ptr(dst, "dst");
    note_write(dst);
    require(op != nullptr, "op is NULL");
    require(n * dtype_bytes(dst_t) <= dst->bytes && n * dtype_bytes(in_t) <= a->bytes &&
                n * dtype_bytes(in_t) <= b->bytes,
            "zip_with: n exceeds a buffer");
    // An f32 input that stands for a deferred cast (a widen of bf16 data, maybe of a deferred
    // narrow) is read from the data it stands for, and the casts need not run.
    const bool wide_ok = in_t == FO_F32 && dst_t == FO_F32;
    const F32Read ra = wide_ok ? f32_read(rt, a, n, dst, true, true) : F32Read{a, 4};
    const F32Read rb = wide_ok ? f32_read(rt, b, n, dst, true, true) : F32Read{b, 4};
    check_buf(ra.buf, "a");
    check_buf(rb.buf, "b");
    if (n == 0) return;
    set_device(rt);
    claim_out(rt, dst, n * dtype_bytes(dst_t));
    TraceScope trace_span(rt, "zip_with");
    if (ra.div != 1 || ra.mod != 0 || rb.div != 1 || rb.mod != 0)
      launch_zip_bcast(rt->stream, dst->ptr, ra.buf->ptr, ra.code, ra.div, ra.mod, ra.pre, rb.buf->ptr, rb.code, rb.div,
                       rb.mod, rb.pre, n, *op);
    else if (ra.code != 4 || rb.code != 4 || ra.pre.n != 0 || rb.pre.n != 0)
      launch_zip_widened(rt->stream, dst->ptr, dst_t, ra.buf->ptr, ra.code, ra.pre, rb.buf->ptr, rb.code, rb.pre, n,
                         *op);
    else
      launch_zip(rt->stream, dst->ptr, dst_t, a->ptr, b->ptr, in_t, n, *op);
  });
}

int32_t fo_zip3_slots(fo_runtime* rt, fo_buffer* dst, const fo_buffer* data, const fo_buffer* port,
                      const fo_buffer* tag_u8, fo_dtype t, uint64_t n, const fo_slots* slots) {
  return guard([&] {
    check_rt(rt);
    check_buf(dst, "dst");
    note_write(dst);
    check_buf(data, "data");
    check_buf(tag_u8, "tag");
    require(slots != nullptr, "slots is NULL");
    require(slots->n_regs >= 0 && slots->n_regs <= 3, "zip3_slots: a pass has 0..3 immediate register slots");
    require(t == FO_F32 || t == FO_I32, "zip3_slots: dtype must be f32 or i32");
    int64_t eb = dtype_bytes(t);
    require(n * eb <= dst->bytes && n * eb <= data->bytes && n <= tag_u8->bytes, "zip3_slots: n exceeds a buffer");
    if (slots->has_port) {
      check_buf(port, "port");
      require(n * eb <= port->bytes, "zip3_slots: n exceeds the port buffer");
    }
    if (n == 0) return;
    set_device(rt);
    TraceScope trace_span(rt, "zip3_slots");
    int32_t* flag = error_word(rt);
    launch_zip3_slots(rt->stream, dst->ptr, data->ptr, slots->has_port ? port->ptr : nullptr,
                      (const uint8_t*)tag_u8->ptr, t, n, *slots, flag);
    rt->err_ops |= 4;
  });
}

int32_t fo_branch_tag(fo_runtime* rt, fo_buffer* tag_u8, const fo_buffer* src, fo_dtype t, uint64_t n,
                      const fo_cmp* cmps) {
  return guard([&] {
    check_rt(rt);
    check_buf(tag_u8, "tag");
    note_write(tag_u8);
    check_buf(src, "src");
    require(cmps != nullptr, "cmps is NULL");
    require(t == FO_F32 || t == FO_I32, "branch_tag: dtype must be f32 or i32");
    require(n <= tag_u8->bytes && n * 4 <= src->bytes, "branch_tag: n exceeds a buffer");
    if (n == 0) return;
    set_device(rt);
    TraceScope trace_span(rt, "branch_tag");
    launch_branch_tag(rt->stream, (uint8_t*)tag_u8->ptr, src->ptr, t, n, cmps);
  });
}

// ---- mapping-driven ops --------------------------------------------------------------------------

}  // extern "C"

namespace {
// The live coordinates of `sym` in `f` (digit weights and counts): `bound` is the largest live
// coordinate plus one (0 when absent); `dense` says whether they fill [0, bound) exactly once.
struct SymCover {
  int64_t bound = 0;
  bool dense = true;
};
SymCover sym_cover(const fm::Factors& f, const std::string& sym) {
  std::vector<const fm::Factor*> ts;
  for (auto& x : f)
    if (x.kind == fm::Factor::Term && x.sym == sym && x.count > 0) ts.push_back(&x);
  SymCover c;
  if (ts.empty()) return c;
  std::sort(ts.begin(), ts.end(), [](const fm::Factor* a, const fm::Factor* b) { return a->weight < b->weight; });
  int64_t expect = 1;
  for (size_t i = 0; i < ts.size(); ++i) {
    if (ts[i]->weight != expect || (i + 1 < ts.size() && ts[i]->count != ts[i]->period)) c.dense = false;
    expect = ts[i]->weight * ts[i]->period;
    c.bound += (ts[i]->count - 1) * ts[i]->weight;
  }
  c.bound += 1;
  return c;
}

// The chain of full-view transposes v[0] -> v[1] -> ... moves each element from its source cell to
// its final cell untouched when every intermediate holds each coordinate the final view reads,
// exactly once and live: then it is the one transpose v[0] -> v.back(). An axis the source lacks is
// a broadcast; an intermediate may lack it too (a transpose cannot drop an axis, so it was added by
// a later step), since no value depends on its coordinate.
bool chain_direct(const std::vector<fm::Factors>& v) {
  const int steps = (int)v.size() - 1;
  bool direct = true;
  for (auto& x : v.back())
    if (x.kind == fm::Factor::Term && direct) {
      const int64_t need = sym_cover(v.back(), x.sym).bound;
      const bool in_src = sym_cover(v[0], x.sym).bound > 0;
      for (int k = 1; k < steps && direct; ++k) {
        const SymCover c = sym_cover(v[k], x.sym);
        direct = c.bound == 0 ? !in_src : (c.dense && c.bound >= need);
      }
    }
  return direct;
}

constexpr int kMaxXposeViews = 8;  // views of one recorded relayout chain

}  // namespace

extern "C" {

int32_t fo_transpose(fo_runtime* rt, fo_buffer* dst, const fo_buffer* src, fo_dtype t, const char* src_view,
                     const char* dst_view, const char* src_map, const char* dst_map, const char* src_offset,
                     const char* dst_offset, int32_t allow_broadcast) {
  return guard([&] {
    check_rt(rt);
    check_ptr(dst, "dst");
    check_ptr(src, "src");
    struct Plan {
      fm::Joint j;
      int64_t dv_size, src_base, dst_base;
    };
    static Memo<Plan> memo;
    const Plan plan = memo.get(
        memo_key({src_view, dst_view, src_map, dst_map, src_offset, dst_offset, allow_broadcast ? "b" : "-"}), [&] {
          fm::Factors sv = flat(src_view, "src_view"), dv = flat(dst_view, "dst_view");
          // transpose_broadcast (backend/op_prep.rs:18-28): the dst leftover after carving out src.
          if (!allow_broadcast)
            require(fm::is_padding(fm::carve(dv, sv)), "transpose: Dst adds axes absent from Src; pass allow_broadcast");
          fm::Joint j = fm::sequence({sv}, {dv}, fm::Mode::Carve);
          fm::Factors sm = src_map && *src_map ? flat(src_map, "src_map") : sv;
          fm::Factors dm = dst_map && *dst_map ? flat(dst_map, "dst_map") : dv;
          return Plan{j, fm::size(dv), fm::window_base(sm, fm::parse_offset_json(src_offset ? src_offset : "")),
                      fm::window_base(dm, fm::parse_offset_json(dst_offset ? dst_offset : ""))};
        });
    const fm::Joint& j = plan.j;
    const int64_t src_base = plan.src_base, dst_base = plan.dst_base;
    if (is_nibble(t)) {  // 4-bit storage, two elements a byte: the one-step form of the nibble chain
      check_buf(src, "src");
      check_buf(dst, "dst");
      note_write(dst);
      const int64_t dst_len = (int64_t)dst->bytes * 2, src_len = (int64_t)src->bytes * 2;
      require(dst_base <= dst_len, "transpose: dst window starts past the buffer");
      const int64_t count = std::min<int64_t>({j.stream_size, plan.dv_size, dst_len - dst_base});
      if (count <= 0) return;
      require(src_base + max_live_offset(j.wheels, 0) < src_len, "transpose: the src window reads past the buffer");
      require(count < (1ll << 31), "transpose: more than 2^31 positions");
      set_device(rt);
      TraceScope trace_span(rt, "transpose");
      const int mem[1] = {0};
      Chain c;
      c.n = 1;
      c.zero_unwritten = 0;
      c.total = (uint32_t)count;
      c.step[0] = ChainStep{to_desc<1>(j.wheels, mem), src_base, (uint32_t)count};
      launch_relayout_chain_nibble(rt->stream, dst->ptr, src->ptr, c, (uint64_t)dst_base);
      return;
    }
    int64_t eb = dtype_bytes(t);
    int64_t dst_len = (int64_t)(dst->bytes / eb), src_len = (int64_t)(src->bytes / eb);
    // A broadcast of f32 data over the whole of dst (every digit live, the src digits one contiguous
    // run from src position 0: dst[i] = src[(i / div) % mod]) is recorded instead of run; a zip
    // reads it through that index map, anything else runs it first (the engine's to_vrf broadcasts
    // of a gain, a RoPE row or a per-row scalar, each read by one zip).
    {
      bool all_live = true;
      for (auto& w : j.wheels) all_live &= w.live == w.size;
      // Innermost first: broadcast digits (stride 0), then one run of consecutive digits whose
      // strides continue each other from 1, then broadcast digits again.
      int64_t place = 1, div = 1, mod = 1;
      int state = 0;  // 0 before the run, 1 in it, 2 after it
      bool pure = all_live;
      for (auto& w : j.wheels) {
        if (w.size > 1) {
          if (w.stride[0] == 0) {
            if (state == 1) state = 2;
          } else if (state == 0 && w.stride[0] == 1) {
            state = 1;
            div = place;
            mod = w.size;
          } else if (state == 1 && w.stride[0] == mod) {
            mod *= w.size;
          } else {
            pure = false;
          }
        }
        place *= w.size;
      }
      const int64_t count = std::min<int64_t>({j.stream_size, plan.dv_size, dst_len - dst_base});
      if (!rt->eager && t == FO_F32 && src != dst && pure && src_base == 0 && dst_base == 0 && count > 0 &&
          count * eb >= (int64_t)dst->bytes && count < (1ll << 31) && mod <= src_len && div < (1ll << 31) &&
          mod < (1ll << 31)) {
        check_filled(src, "src");
        set_device(rt);
        claim_out(rt, dst, dst->bytes);
        note_write(dst);
        const int mem[1] = {0};
        std::lock_guard<std::mutex> lock(g_widen_mu);
        WidenRecord r{dst, src, FO_F32, (uint64_t)count, FO_F32, fo_op{}, rt, true};
        r.kind = 1;
        r.div = (uint32_t)div;
        r.mod = (uint32_t)mod;
        r.wheels = to_desc<1>(j.wheels, mem);
        g_widen.push_back(r);
        dst->widen_pending = true;
        return;
      }
    }
    // A relayout that writes the whole of dst (the dst view is the buffer's size; no window or map),
    // from a source with nothing deferred into it, or from a recorded relayout read with that
    // relayout's own last view, is recorded instead of run. Consecutive relayouts -- the engine's
    // fetch, switch, collect and commit, each into a fresh storage (tensor/mod.rs:302-306) --
    // compose into one pass while the chain keeps the direct form, and run when anything else reads
    // them (or their source is written). The intermediates' records stay for any other reader.
    const bool plain = !(src_offset && *src_offset) && !(dst_offset && *dst_offset) && !(src_map && *src_map) &&
                       !(dst_map && *dst_map);
    if (!rt->eager && plain && src != dst && src_base == 0 && dst_base == 0 &&
        plan.dv_size * eb == (int64_t)dst->bytes) {
      std::vector<std::string> views;
      WidenRecord xr{};
      const bool compose = deferred_xpose(rt, src, &xr) && xr.xt == t && xr.views.back() == src_view &&
                           xr.src != dst && (int)xr.views.size() < kMaxXposeViews;
      if (compose) {
        views = xr.views;
        views.push_back(dst_view);
      } else if (!src->widen_pending) {
        views = {src_view, dst_view};
      }
      struct XPlan {
        bool ok;
        fm::Joint j;
        int64_t count;
      };
      static Memo<XPlan> xmemo;
      std::string key;
      for (auto& v : views) key += v + '\x02';
      const XPlan xp = views.empty() ? XPlan{false, {}, 0} : xmemo.get(key, [&] {
        std::vector<fm::Factors> v;
        for (auto& x : views) v.push_back(flat(x.c_str(), "view"));
        if (!chain_direct(v)) return XPlan{false, {}, 0};
        fm::Joint jj = views.size() == 2 ? j : fm::sequence({v[0]}, {v.back()}, fm::Mode::Carve);
        return XPlan{true, jj, std::min<int64_t>(jj.stream_size, fm::size(v.back()))};
      });
      const fo_buffer* s0 = compose ? xr.src : src;
      if (xp.ok && xp.count > 0 && xp.count < (1ll << 31) &&
          max_live_offset(xp.j.wheels, 0) < (int64_t)(s0->bytes / eb)) {
        check_filled(s0, "src");
        set_device(rt);
        bool live = true;
        for (auto& w : xp.j.wheels) live &= w.live == w.size;
        if (live && xp.count * eb >= (int64_t)dst->bytes) {  // every byte written
          note_overwrite(dst);
          claim_out(rt, dst, dst->bytes);
        } else {
          note_write(dst);  // the dead cells keep what dst holds
        }
        const int mem[1] = {0};
        std::lock_guard<std::mutex> lock(g_widen_mu);
        WidenRecord r{dst, s0, t, (uint64_t)xp.count, t, fo_op{}, rt, true};
        r.kind = 3;
        r.views = std::move(views);
        r.xt = t;
        r.count = xp.count;
        r.wheels = to_desc<1>(xp.j.wheels, mem);
        g_widen.push_back(std::move(r));
        dst->widen_pending = true;
        return;
      }
    }
    // An f32 source that is a still-deferred widen of bf16 data may be read from that data.
    WidenRecord wsrc{};
    const bool narrow = t == FO_F32 && src != dst &&
                        deferred_bf16_widen(rt, src, (uint64_t)(src_base + max_live_offset(j.wheels, 0) + 1), &wsrc) &&
                        wsrc.src != dst;
    check_buf(narrow ? wsrc.src : src, "src");
    require(dst_base <= dst_len, "transpose: dst window starts past the buffer");
    int64_t count = std::min<int64_t>({j.stream_size, plan.dv_size, dst_len - dst_base});
    // dst positions dst_base .. dst_base + count - 1 are written where every digit is live: from
    // position 0 over the whole buffer with no dead digit, the op overwrites every byte and a
    // pending zero fill is not needed; otherwise the fill goes first.
    bool all_live = true;
    for (auto& w : j.wheels) all_live &= w.live == w.size;
    // A fresh storage written in part from position 0 (a padded layout): one pass writes the live
    // cells and zero everywhere else the pending fill would have.
    const uint64_t cap = (dst->capacity + 15) & ~15ull;
    const bool fused_fill = count > 0 && dst_base == 0 && !narrow && dst->zero_pending && !dst->widen_pending &&
                            cap % (uint64_t)eb == 0 && cap / (uint64_t)eb < (1ull << 31) &&
                            !(all_live && count * eb >= (int64_t)dst->bytes);
    if (count > 0 && dst_base == 0 && all_live && count * eb >= (int64_t)dst->bytes) {
      set_device(rt);
      claim_out(rt, dst, dst->bytes);
    } else if (!fused_fill) {
      check_buf(dst, "dst");
    }
    note_write(dst);
    if (count <= 0) return;
    require(src_base + max_live_offset(j.wheels, 0) < src_len, "transpose: the src window reads past the buffer");
    require(count < (1ll << 31), "transpose: more than 2^31 positions");
    set_device(rt);
    TraceScope trace_span(rt, "transpose");
    const int mem[1] = {0};
    const Wheels<1> w = to_desc<1>(j.wheels, mem);
    if (fused_fill) {
      Chain c;
      c.n = 1;
      c.zero_unwritten = 1;
      c.total = (uint32_t)(cap / (uint64_t)eb);
      c.step[0] = ChainStep{w, src_base, (uint32_t)count};
      mark_filled(dst);
      launch_relayout_chain(rt->stream, dst->ptr, src->ptr, eb, c);
      return;
    }
    if (narrow && launch_relayout_widen(rt->stream, (float*)dst->ptr, (const uint16_t*)wsrc.src->ptr, dst_base, src_base,
                                        count, w))
      return;
    if (narrow) check_buf(src, "src");  // no widening form for this layout: the cast runs first
    launch_relayout(rt->stream, dst->ptr, src->ptr, eb, dst_base, src_base, count, w);
  });
}

int32_t fo_transpose_chain(fo_runtime* rt, fo_buffer* dst, const fo_buffer* src, fo_dtype t, int32_t n_views,
                           const char* const* views, const int32_t* allow_broadcast) {
  return guard([&] {
    check_rt(rt);
    check_buf(dst, "dst");
    note_write(dst);
    check_buf(src, "src");
    require(n_views >= 2 && views != nullptr, "transpose_chain: needs at least two views");
    const bool nib = is_nibble(t);                 // 4-bit storage: two elements a byte
    const int64_t eb = nib ? 1 : dtype_bytes(t);
    auto elems = [&](const fo_buffer* b) { return nib ? (int64_t)b->bytes * 2 : (int64_t)(b->bytes / eb); };
    std::vector<fm::Factors> v;
    for (int i = 0; i < n_views; ++i) v.push_back(flat(views[i], "views[i]"));
    const int steps = n_views - 1;
    bool any_broadcast = false;
    std::vector<ChainStep> cs(steps);
    for (int k = 0; k < steps; ++k) {
      const bool bc = allow_broadcast && allow_broadcast[k];
      any_broadcast |= bc;
      if (!bc)
        require(fm::is_padding(fm::carve(v[k + 1], v[k])),
                "transpose_chain: step " + std::to_string(k) + " adds axes absent from its source; allow its broadcast");
      fm::Joint j = fm::sequence({v[k]}, {v[k + 1]}, fm::Mode::Carve);
      const int64_t src_len = k == 0 ? elems(src) : fm::size(v[k]);
      const int64_t dst_len = k == steps - 1 ? elems(dst) : fm::size(v[k + 1]);
      const int64_t count = std::max<int64_t>(0, std::min<int64_t>({j.stream_size, fm::size(v[k + 1]), dst_len}));
      require(max_live_offset(j.wheels, 0) < src_len || count == 0,
              "transpose_chain: step " + std::to_string(k) + " reads past its source");
      require(fm::size(v[k + 1]) < (1ll << 31), "transpose_chain: a view of more than 2^31 positions");
      const int mem[1] = {0};
      cs[k].w = to_desc<1>(j.wheels, mem);
      cs[k].src_base = 0;
      cs[k].count = (uint32_t)count;
    }
    if (cs[steps - 1].count == 0) return;
    set_device(rt);
    TraceScope trace_span(rt, "transpose_chain");

    // Direct form (chain_direct): the one transpose first view -> last view, with that kernel's
    // tiled and 16-byte paths.
    if (chain_direct(v)) {
      if (!any_broadcast) require(fm::is_padding(fm::carve(v.back(), v[0])), "transpose_chain: broadcast mismatch");
      fm::Joint j = fm::sequence({v[0]}, {v.back()}, fm::Mode::Carve);
      const int64_t count = std::min<int64_t>({j.stream_size, fm::size(v.back()), elems(dst)});
      require(max_live_offset(j.wheels, 0) < elems(src), "transpose_chain: reads past the source");
      const int mem[1] = {0};
      if (nib) {
        if (count <= 0) return;
        Chain c;
        c.n = 1;
        c.zero_unwritten = 0;
        c.total = (uint32_t)count;
        c.step[0] = ChainStep{to_desc<1>(j.wheels, mem), 0, (uint32_t)count};
        launch_relayout_chain_nibble(rt->stream, dst->ptr, src->ptr, c, 0);
        return;
      }
      launch_relayout(rt->stream, dst->ptr, src->ptr, eb, 0, 0, count, to_desc<1>(j.wheels, mem));
      return;
    }

    // General form: groups of up to kMaxChain steps, each a back-walking gather; a group that ends
    // on an intermediate materializes it (whole, zero where unwritten) in scratch.
    const void* in = src->ptr;
    int k0 = 0;
    uint8_t* sc = nullptr;
    uint64_t half = 0;
    int flip = 0;
    while (k0 < steps) {
      const int k1 = std::min(steps, k0 + kMaxChain);
      Chain c;
      c.n = k1 - k0;
      for (int k = k0; k < k1; ++k) c.step[k - k0] = cs[k];
      void* out;
      if (k1 == steps) {
        c.total = cs[steps - 1].count;
        c.zero_unwritten = 0;
        out = dst->ptr;
      } else {
        if (!sc) {
          int64_t most = 0;
          for (int k = 1; k < steps; ++k) most = std::max(most, fm::size(v[k]));
          half = ((nib ? (uint64_t)(most + 1) / 2 : (uint64_t)most * eb) + 255) & ~(uint64_t)255;
          sc = (uint8_t*)runtime_scratch(rt, 2 * half);
        }
        c.total = (uint32_t)fm::size(v[k1]);
        c.zero_unwritten = 1;
        out = sc + (flip ? half : 0);
        flip ^= 1;
      }
      if (nib)
        launch_relayout_chain_nibble(rt->stream, out, in, c, 0);
      else
        launch_relayout_chain(rt->stream, out, in, eb, c);
      in = out;
      k0 = k1;
    }
  });
}

int32_t fo_transmute(fo_runtime* rt, fo_buffer* dst, const fo_buffer* src, fo_dtype t, const char* src_map,
                     const char* dst_map) {
  return guard([&] {
    check_rt(rt);
    check_buf(dst, "dst");
    note_write(dst);
    check_buf(src, "src");
    fm::Factors sm = flat(src_map, "src_map"), dm = flat(dst_map, "dst_map");
    int64_t eb = dtype_bytes(t);
    int64_t dn = fm::size(dm);
    require(dn * eb <= (int64_t)dst->bytes, "transmute: dst buffer smaller than dst_map");
    require(fm::size(sm) * eb <= (int64_t)src->bytes, "transmute: src buffer smaller than src_map");
    // Self-walks: wire position <-> live rank.
    auto self = [](const fm::Factors& f, bool by_live) {
      std::vector<fm::Wheel> ws;
      auto st = fm::strides(f);
      for (size_t i = f.size(); i-- > 0;) {
        fm::Wheel w;
        w.size = by_live ? f[i].count : f[i].extent;
        w.live = f[i].count;
        w.stride = {st[i]};
        ws.push_back(w);
      }
      return ws;
    };
    auto dw = self(dm, false), sw = self(sm, true);
    int64_t dlive = 1, slive = 1;
    for (auto& x : dm) dlive *= x.count;
    for (auto& x : sm) slive *= x.count;
    require(slive >= dlive, "transmute: dst_map has more live elements than src_map");
    if (dn == 0) return;
    require(dn < (1ll << 31), "transmute: more than 2^31 positions");
    set_device(rt);
    TraceScope trace_span(rt, "transmute");
    const int mem[1] = {0};
    launch_transmute(rt->stream, dst->ptr, src->ptr, eb, dn, to_desc<1>(dw, mem), to_desc<1>(sw, mem));
  });
}

int32_t fo_scatter(fo_runtime* rt, fo_buffer* dst, const fo_buffer* src, const fo_buffer* index, fo_dtype t,
                   const char* src_map, const char* key_map, const char* dst_map, const char* idx_map,
                   int32_t scaled) {
  return guard([&] {
    check_rt(rt);
    check_buf(dst, "dst");
    note_write(dst);
    check_buf(src, "src");
    check_buf(index, "index");
    fm::Factors sm = flat(src_map, "src_map"), km = flat(key_map, "key_map"), dm = flat(dst_map, "dst_map"),
                im = flat(idx_map, "idx_map");
    // scatter_params (backend/op_prep.rs:45-54): payload = Src / Key; the indexed dst axis is the
    // first live axis of Dst / payload.
    fm::Factors payload = fm::remove_padding(fm::carve(sm, km));
    fm::Factors axis;
    try {
      axis = fm::first_axis(fm::carve(dm, payload));
    } catch (const fm::Error&) {
      throw InvalidArg("scatter: dst residue has no live target axis");
    }
    const int64_t eb = dtype_bytes(t), keys = fm::size(km), axis_size = fm::size(axis), np = fm::size(payload);
    require(fm::size(im) >= keys, "scatter: the index tensor has fewer cells than the key");
    require((int64_t)index->bytes >= keys * 4, "scatter: index buffer shorter than the key");
    auto ws = stream_wheels(sm, payload, km, "scatter src");
    auto wd = stream_wheels(dm, payload, axis, "scatter dst");
    require(max_live_offset(ws, 0) < (int64_t)(src->bytes / eb), "scatter: src reads past the buffer");
    require(max_live_offset(wd, 0) < (int64_t)(dst->bytes / eb), "scatter: dst writes past the buffer");
    require(np * keys < (1ll << 31) && np * axis_size < (1ll << 31), "scatter: more than 2^31 positions");
    // decode_stride (buf.rs:816-822): a scaled index is a byte offset of payload-sized blocks.
    const int64_t div = scaled ? np * eb : 1;
    require(div < (1ll << 31), "scatter: payload block too large");
    if (np * keys == 0) return;
    set_device(rt);
    TraceScope trace_span(rt, "scatter");
    int32_t* flag = error_word(rt);
    // Winner words: grown (and zeroed) when too short, and zeroed again when the 32-bit generation
    // wraps; otherwise each call only takes the next generation. A recorded scatter has words of its
    // own, cleared by a kernel in the graph, so every launch starts from a clean generation. One key
    // slot (a cache row append) writes no target twice and needs none: the copy checks the index.
    uint64_t* win = nullptr;
    uint32_t gen = 0;
    if (keys > 1) {
      if (recording(rt)) {
        auto blk = take_block(rt, (uint64_t)axis_size * 8);
        launch_zero(rt->stream, blk.first, blk.second);
        win = (uint64_t*)blk.first;
        gen = 1;
      } else if (rt->scatter_win_slots < (uint64_t)axis_size || rt->scatter_gen == UINT32_MAX) {
        FO_HIP(hipStreamSynchronize(rt->stream));
        if (rt->scatter_win_slots < (uint64_t)axis_size) {
          if (rt->scatter_win) FO_HIP(hipFree(rt->scatter_win));
          rt->scatter_win = nullptr;
          rt->scatter_win_slots = 0;
          FO_HIP(hipMalloc((void**)&rt->scatter_win, (size_t)axis_size * 8));
          rt->scatter_win_slots = (uint64_t)axis_size;
        }
        FO_HIP(hipMemsetAsync(rt->scatter_win, 0, (size_t)rt->scatter_win_slots * 8, rt->stream));
        rt->scatter_gen = 0;
      }
      if (!gen) {
        gen = ++rt->scatter_gen;
        win = rt->scatter_win;
      }
    }
    const int mem[1] = {0};
    launch_scatter(rt->stream, dst->ptr, src->ptr, (const int32_t*)index->ptr, eb, np, keys, axis_size, (int32_t)div,
                   to_desc<1>(ws, mem), to_desc<1>(wd, mem), inner_part_wheels(ws), inner_part_wheels(wd), win, gen,
                   flag);
    rt->err_ops |= 2;
  });
}

int32_t fo_gather(fo_runtime* rt, fo_buffer* dst, const fo_buffer* src, const fo_buffer* index, fo_dtype t,
                  const char* src_map, const char* dst_map, const char* idx_map, int32_t scaled) {
  return guard([&] {
    check_rt(rt);
    check_buf(dst, "dst");
    note_write(dst);
    check_buf(src, "src");
    check_buf(index, "index");
    fm::Factors sm = flat(src_map, "src_map"), dm = flat(dst_map, "dst_map"), im = flat(idx_map, "idx_map");
    // gather_params (backend/op_prep.rs:78-89): payload = Dst / Idx; the indexed (table) axis is
    // the first live axis of Src / payload; the dst slots are the index tensor's own mapping.
    fm::Factors payload = fm::remove_padding(fm::carve(dm, im));
    fm::Factors axis;
    try {
      axis = fm::first_axis(fm::carve(sm, payload));
    } catch (const fm::Error&) {
      throw InvalidArg("gather: src residue has no live target axis");
    }
    const int64_t eb = dtype_bytes(t), slots = fm::size(im), axis_size = fm::size(axis), np = fm::size(payload);
    require((int64_t)index->bytes >= slots * 4, "gather: index buffer shorter than the index mapping");
    auto ws = stream_wheels(sm, payload, axis, "gather src");
    auto wd = stream_wheels(dm, payload, im, "gather dst");
    require(max_live_offset(ws, 0) < (int64_t)(src->bytes / eb), "gather: src reads past the buffer");
    require(max_live_offset(wd, 0) < (int64_t)(dst->bytes / eb), "gather: dst writes past the buffer");
    require(np * slots < (1ll << 31) && np * axis_size < (1ll << 31), "gather: more than 2^31 positions");
    const int64_t div = scaled ? np * eb : 1;
    require(div < (1ll << 31), "gather: payload block too large");
    if (np * slots == 0) return;
    set_device(rt);
    TraceScope trace_span(rt, "gather");
    int32_t* flag = error_word(rt);
    const int mem[1] = {0};
    launch_gather(rt->stream, dst->ptr, src->ptr, (const int32_t*)index->ptr, eb, np, slots, axis_size, (int32_t)div,
                  to_desc<1>(ws, mem), to_desc<1>(wd, mem), inner_part_wheels(ws), inner_part_wheels(wd), flag);
    rt->err_ops |= 1;
  });
}

int32_t fo_reduce(fo_runtime* rt, fo_buffer* dst, const fo_buffer* src, fo_dtype t, const char* src_map,
                  const char* dst_map, int32_t op, uint32_t identity, int32_t allow_broadcast) {
  return guard([&] {
    check_rt(rt);
    check_ptr(dst, "dst");
    note_write(dst);
    check_ptr(src, "src");
    require(t == FO_F32 || t == FO_I32 || t == FO_BF16, "reduce: dtype must be f32, i32 or bf16");
    require(op >= FO_RED_ADD && op <= FO_RED_ADD_SAT, "reduce: unknown op");
    require(op != FO_RED_ADD_SAT || t == FO_I32, "reduce: saturating add is i32 only");
    struct Plan {
      int64_t out_count;
      std::vector<fm::Wheel> ow, rw;
    };
    static Memo<Plan> memo;
    const Plan plan = memo.get(memo_key({src_map, dst_map, allow_broadcast ? "b" : "-"}), [&] {
      fm::Factors s = flat(src_map, "src_map"), d = flat(dst_map, "dst_map");
      // BufStorage::reduce (buf.rs:331-376): inter = dst.carve(broadcast), residue = src.carve(inter).
      auto bsyms = fm::broadcast_symbols(s, d);
      require(allow_broadcast || bsyms.empty(),
              "reduce: Dst adds axes absent from the source; pass allow_broadcast=true for reduce-then-broadcast");
      fm::Factors bcast;
      for (auto& x : d)
        if (x.kind == fm::Factor::Term && std::find(bsyms.begin(), bsyms.end(), x.sym) != bsyms.end())
          bcast.push_back(x);
      fm::Factors inter = bcast.empty() ? d : fm::carve(d, bcast);
      fm::Factors residue = fm::carve(s, inter);
      fm::Joint j = fm::sequence({s}, {d, residue}, fm::Mode::Read);
      return Plan{fm::size(d), part(j, 0), live_only(part(j, 1))};
    });
    const std::vector<fm::Wheel>& ow = plan.ow;
    const std::vector<fm::Wheel>& rw = plan.rw;
    int64_t eb = dtype_bytes(t);
    int64_t out_count = plan.out_count;
    require(out_count * eb <= (int64_t)dst->bytes, "reduce: dst buffer smaller than dst_map");
    require(out_count < (1ll << 31), "reduce: more than 2^31 output cells");
    if (out_count == 0) return;
    set_device(rt);
    const int mem[1] = {0};
    const Wheels<1> owd = to_desc<1>(ow, mem), rwd = to_desc<1>(rw, mem);
    const int64_t src_len = (int64_t)(src->bytes / eb);
    const ReduceSplit split = plan_reduce_split(t, op, src->ptr, src_len, out_count, owd, rwd);
    // An f32 source that stands for a deferred widen of bf16 data (covering the whole buffer), maybe
    // of a deferred narrow, is read from the data it stands for, unless the two-pass column form is
    // chosen.
    const F32Read rs = t == FO_F32 && split.nchunks == 0 && src != dst ? f32_read(rt, src, (uint64_t)src_len, dst)
                                                                        : F32Read{src, 4};
    check_buf(rs.buf, "src");
    claim_out(rt, dst, (uint64_t)(out_count * eb));  // every cell is written, a dead one with the identity
    TraceScope trace_span(rt, "reduce");
    if (rs.code != 4)
      launch_reduce_widened(rt->stream, dst->ptr, rs.buf->ptr, rs.code == kReadViaBf16, src_len, out_count, owd, rwd,
                            op, identity);
    else if (split.nchunks > 0)
      launch_reduce_split(rt->stream, dst->ptr, src->ptr, t, out_count, owd, rwd, op, identity, split,
                          runtime_scratch(rt, split.scratch_bytes));
    else
      launch_reduce(rt->stream, dst->ptr, src->ptr, t, src_len, out_count, owd, rwd, op, identity);
  });
}

}  // extern "C"

namespace {

// Backend::contraction behind both entry points. `noalloc`: working memory (the i4 unpack and the
// i32 staging of an i4 result) comes from the static scratch instead of the runtime's, so the call
// allocates no device memory.
void contraction_impl(fo_runtime* rt, fo_buffer* out, const fo_buffer* lhs, const fo_buffer* rhs, fo_dtype in_t,
                      fo_dtype out_t, const char* lhs_map, const char* rhs_map, const char* pre_reduce,
                      const char* out_map, bool noalloc) {
  {
    check_rt(rt);
    check_ptr(out, "out");
    note_write(out);
    // The operands are checked here and made current (zero fill, deferred cast) below, unless the
    // contraction reads their narrow sources.
    check_ptr(lhs, "lhs");
    check_ptr(rhs, "rhs");
    bool ok_types = (in_t == FO_BF16 && (out_t == FO_BF16 || out_t == FO_F32)) ||
                    (in_t == FO_I8 && (out_t == FO_I8 || out_t == FO_I32)) || (in_t == FO_F32 && out_t == FO_F32) ||
                    (in_t == FO_I32 && out_t == FO_I32) ||
                    ((in_t == FO_F8E4M3 || in_t == FO_F8E5M2) && (out_t == in_t || out_t == FO_F32)) ||
                    (in_t == FO_I4 && (out_t == FO_I4 || out_t == FO_I32));
    require(ok_types, "contraction: unsupported operand/output dtype pair");
    // contraction_in (buf.rs:401-447): contracted = pre_reduce.carve(out); one ReadPlan per operand.
    struct Plan {
      int64_t l_size, r_size, out_count;
      std::vector<fm::Wheel> ow, rw;
    };
    static Memo<Plan> memo;
    const Plan plan = memo.get(memo_key({lhs_map, rhs_map, pre_reduce, out_map}), [&] {
      fm::Factors l = flat(lhs_map, "lhs_map"), r = flat(rhs_map, "rhs_map");
      fm::Factors pre = flat(pre_reduce, "pre_reduce"), o = flat(out_map, "out_map");
      fm::Factors contracted = fm::carve(pre, o);
      fm::Joint j = fm::sequence({l, r}, {o, contracted}, fm::Mode::Read);
      return Plan{fm::size(l), fm::size(r), fm::size(o), merge_contiguous(part(j, 0)),
                  merge_contiguous(live_only(part(j, 1)))};
    });
    const std::vector<fm::Wheel>& ow = plan.ow;
    const std::vector<fm::Wheel>& rw = plan.rw;
    int64_t out_count = plan.out_count;
    require(span_bytes(out_t, (uint64_t)out_count) <= out->bytes, "contraction: out buffer smaller than out_map");
    require(out_count < (1ll << 31), "contraction: more than 2^31 output cells");
    require(out_t != FO_I4 || out_count % 2 == 0, "contraction: a 4-bit output stream needs an even cell count");
    if (out_count == 0) return;
    set_device(rt);
    TraceScope trace_span(rt, "contraction");

    // i4 operands (ContractionCast for i4: widen to i32, cast.rs:365-367) are unpacked to one i8 per
    // element in scratch, exactly, and contracted as i8; an i4 result is computed as i32 and packed
    // (one narrow per cell, Cast<i4> for i32).
    fo_dtype ct = in_t, co = out_t;
    const void *L = lhs->ptr, *R = rhs->ptr;
    void* O = out->ptr;
    int64_t lhs_len, rhs_len;
    WidenRecord wl{}, wr{};
    const bool narrow = !rt->eager && (in_t == FO_F32 || in_t == FO_I32) && out_t == in_t && find_widen(lhs, &wl) &&
                        find_widen(rhs, &wr) && wl.src_t == wr.src_t && (int64_t)wl.n >= plan.l_size &&
                        (int64_t)wr.n >= plan.r_size;
    if (!narrow) {
      check_buf(lhs, "lhs");
      check_buf(rhs, "rhs");
    }
    // A GEMV's x given as a deferred narrow of f32 data is read from that data (rounded as it is
    // staged); any other kernel below runs the narrow first.
    WidenRecord xr{};
    const bool x_narrowed = narrow && deferred_bf16_narrow(rt, wl.src, wl.n, &xr) && xr.src != out;
    if (narrow) {  // the narrow sources, made current (a deferred narrow into one runs here)
      check_buf(x_narrowed ? xr.src : wl.src, "lhs");
      check_buf(wr.src, "rhs");
    }
    if (in_t == FO_I4) {
      auto up = [](uint64_t v) { return (v + 255) & ~(uint64_t)255; };
      const uint64_t la = up(lhs->bytes * 2), ra = up(rhs->bytes * 2), oa = out_t == FO_I4 ? (uint64_t)out_count * 4 : 0;
      uint8_t* sc = noalloc ? (uint8_t*)static_scratch(rt, la + ra + oa, "contraction_noalloc")
                            : (uint8_t*)runtime_scratch(rt, la + ra + oa);
      launch_unpack_i4(rt->stream, (int8_t*)sc, lhs->ptr, lhs->bytes);
      launch_unpack_i4(rt->stream, (int8_t*)(sc + la), rhs->ptr, rhs->bytes);
      L = sc;
      R = sc + la;
      ct = FO_I8;
      if (out_t == FO_I4) {
        co = FO_I32;
        O = sc + la + ra;
      }
      lhs_len = (int64_t)lhs->bytes * 2;
      rhs_len = (int64_t)rhs->bytes * 2;
    } else if (narrow) {
      // contraction_prewidened of two widened operands: contract their narrow sources (the
      // pending-widen records above), accumulating in the same type.
      ct = wl.src_t;
      L = wl.src->ptr;
      R = wr.src->ptr;
      lhs_len = (int64_t)wl.n;
      rhs_len = (int64_t)wr.n;
    } else {
      lhs_len = (int64_t)(lhs->bytes / dtype_bytes(in_t));
      rhs_len = (int64_t)(rhs->bytes / dtype_bytes(in_t));
    }

    auto run = [&] {
      // Out wheels split into rows (read by lhs only, or by neither operand: repeated rows),
      // columns (rhs only) and batch cells (both), with the place of each in the dense out stream.
      struct Part {
        fm::Wheel w;
        int64_t place;
      };
      std::vector<Part> mw, nw, bw;
      bool padded = false;
      int64_t place = 1;
      for (auto& w : ow) {
        padded |= w.live != w.size;
        const bool la = w.stride[0] != 0, rb = w.stride[1] != 0;
        (la && rb ? bw : (!la && rb) ? nw : mw).push_back({w, place});
        place *= w.size;
      }
      const bool unit_k = rw.size() == 1 && rw[0].stride[0] == 1 && rw[0].stride[1] == 1;
      // One lhs vector against contiguous rhs rows (a token against a weight matrix): the GEMV
      // kernel, one lane folding each cell in k order.
      if (unit_k && mw.empty() && bw.empty() && nw.size() == 1 && !padded) {
        const int64_t N = nw[0].w.size, K = rw[0].size, ldw = nw[0].w.stride[1];
        if (K - 1 < lhs_len && (N - 1) * ldw + K - 1 < rhs_len && gemv_supported(ct, co, L, R, N, K, ldw)) {
          const bool xf = x_narrowed && gemv_takes_f32_x(K);
          if (x_narrowed && !xf) check_buf(wl.src, "lhs");
          launch_gemv(rt->stream, O, xf ? xr.src->ptr : L, R, ct, co, N, K, ldw, nw[0].place, xf);
          return;
        }
      }
      if (x_narrowed) check_buf(wl.src, "lhs");
      // Batched dot products (out wheels read both operands, or the rhs only, or neither: padding;
      // a batch of GEMVs such as a lane-broadcast TRF contraction per slice): one lane folds each
      // cell's two rows in k order.
      const bool rows_repeat_only =
          std::all_of(mw.begin(), mw.end(), [](const Part& p) { return p.w.stride[0] == 0 && p.w.stride[1] == 0; });
      if (unit_k && rows_repeat_only && !bw.empty()) {
        const int64_t K = rw[0].size;
        if (max_live_offset(ow, 0) + K - 1 < lhs_len && max_live_offset(ow, 1) + K - 1 < rhs_len) {
          const int64_t eb = dtype_bytes(ct);
          bool vec = ((uintptr_t)L % 16) == 0 && ((uintptr_t)R % 16) == 0;
          for (auto& w : ow) vec &= (w.stride[0] * eb) % 16 == 0 && (w.stride[1] * eb) % 16 == 0;
          const int mem[2] = {0, 1};
          if (launch_contraction_dot(rt->stream, O, L, R, ct, co, out_count, to_desc<2>(ow, mem), K, vec)) return;
        }
      }
      if (gemm_supported(ct, co) && unit_k) {
        // The tiled kernel: one affine row, column and batch wheel each, no padding.
        if (!padded && mw.size() <= 1 && nw.size() <= 1 && bw.size() <= 1) {
          GemmDesc d;
          d.M = mw.empty() ? 1 : mw[0].w.size;
          d.N = nw.empty() ? 1 : nw[0].w.size;
          d.K = rw[0].size;
          d.batch = bw.empty() ? 1 : bw[0].w.size;
          d.lda = mw.empty() ? 0 : mw[0].w.stride[0];
          d.ldb = nw.empty() ? 0 : nw[0].w.stride[1];
          d.ldc_m = mw.empty() ? 0 : mw[0].place;
          d.ldc_n = nw.empty() ? 0 : nw[0].place;
          d.a_batch = bw.empty() ? 0 : bw[0].w.stride[0];
          d.b_batch = bw.empty() ? 0 : bw[0].w.stride[1];
          d.c_batch = bw.empty() ? 0 : bw[0].place;
          int64_t amax = (d.batch - 1) * d.a_batch + (d.M - 1) * d.lda + d.K - 1;
          int64_t bmax = (d.batch - 1) * d.b_batch + (d.N - 1) * d.ldb + d.K - 1;
          if (amax < lhs_len && bmax < rhs_len && gemm_aligned(L, R, ct, d)) {
            launch_gemm(rt->stream, O, L, R, ct, co, d, rt->gemm_ws);
            return;
          }
          if (amax < lhs_len && bmax < rhs_len && launch_gemm_any(rt->stream, O, L, R, ct, co, d, rt->gemm_ws)) return;
        }
        // The wheel-decoded kernel: rows, columns and batch cells over any number of wheels
        // (live digits only; dead out cells zeroed first), when a 32 x 32 tile is at least a
        // quarter used and every read stays inside the operands.
        int64_t M = 1, N = 1, B = 1, amax = rw[0].size - 1, bmax = rw[0].size - 1, align = rw[0].size;
        auto gcd = [](int64_t x, int64_t y) {
          while (y) {
            int64_t t = x % y;
            x = y;
            y = t;
          }
          return x;
        };
        for (auto& p : mw) M *= p.w.live, amax += (p.w.live - 1) * p.w.stride[0], align = gcd(align, p.w.stride[0]);
        for (auto& p : nw) N *= p.w.live, bmax += (p.w.live - 1) * p.w.stride[1], align = gcd(align, p.w.stride[1]);
        for (auto& p : bw) {
          B *= p.w.live;
          amax += (p.w.live - 1) * p.w.stride[0];
          bmax += (p.w.live - 1) * p.w.stride[1];
          align = gcd(gcd(align, p.w.stride[0]), p.w.stride[1]);
        }
        const int nwheels_ok = (int)std::max({mw.size(), nw.size(), bw.size()}) <= kMaxWheels;
        if (nwheels_ok && M >= 8 && N >= 8 && amax < lhs_len && bmax < rhs_len &&
            gemm_wheels_supported(ct, co, rw[0].size, align)) {
          Wheels<2> dm{}, dn{};
          Wheels<3> db{};
          auto fill2 = [](Wheels<2>& d, const std::vector<Part>& ps, int k) {
            for (auto& p : ps) {
              if (p.w.live <= 1) continue;
              const int i = d.n++;
              d.size[i] = d.live[i] = (uint32_t)p.w.live;
              d.div[i] = FastDiv((uint32_t)p.w.live);
              d.stride[0][i] = p.w.stride[k];
              d.stride[1][i] = p.place;
            }
          };
          fill2(dm, mw, 0);
          fill2(dn, nw, 1);
          for (auto& p : bw) {
            if (p.w.live <= 1) continue;
            const int i = db.n++;
            db.size[i] = db.live[i] = (uint32_t)p.w.live;
            db.div[i] = FastDiv((uint32_t)p.w.live);
            db.stride[0][i] = p.w.stride[0];
            db.stride[1][i] = p.w.stride[1];
            db.stride[2][i] = p.place;
          }
          if (padded) launch_zero(rt->stream, O, span_bytes(co, (uint64_t)out_count));
          launch_gemm_wheels(rt->stream, O, L, R, ct, co, M, N, rw[0].size, B, dm, dn, db);
          return;
        }
      }
      // One row, column, batch and contracted wheel each, no padding, and no MFMA form above (f32 and
      // i32 operands, or K strided, or fewer than 8 rows or columns): the vector-unit tile kernel,
      // each cell folded in k order (any k strides).
      if (!padded && rw.size() == 1 && mw.size() <= 1 && nw.size() <= 1 && bw.size() <= 1) {
        GemmDesc d;
        d.M = mw.empty() ? 1 : mw[0].w.size;
        d.N = nw.empty() ? 1 : nw[0].w.size;
        d.K = rw[0].size;
        d.batch = bw.empty() ? 1 : bw[0].w.size;
        d.lda = mw.empty() ? 0 : mw[0].w.stride[0];
        d.ldb = nw.empty() ? 0 : nw[0].w.stride[1];
        d.ldc_m = mw.empty() ? 0 : mw[0].place;
        d.ldc_n = nw.empty() ? 0 : nw[0].place;
        d.a_batch = bw.empty() ? 0 : bw[0].w.stride[0];
        d.b_batch = bw.empty() ? 0 : bw[0].w.stride[1];
        d.c_batch = bw.empty() ? 0 : bw[0].place;
        const int64_t sa = rw[0].stride[0], sb = rw[0].stride[1];
        const int64_t amax = (d.batch - 1) * d.a_batch + (d.M - 1) * d.lda + (d.K - 1) * sa;
        const int64_t bmax = (d.batch - 1) * d.b_batch + (d.N - 1) * d.ldb + (d.K - 1) * sb;
        if (amax < lhs_len && bmax < rhs_len && launch_contraction_simt(rt->stream, O, L, R, ct, co, d, sa, sb)) return;
      }
      const int mem[2] = {0, 1};
      launch_contraction_generic(rt->stream, O, L, R, ct, co, lhs_len, rhs_len, out_count, to_desc<2>(ow, mem),
                                 to_desc<2>(rw, mem));
    };
    claim_out(rt, out, span_bytes(out_t, (uint64_t)out_count));  // every cell is written
    run();
    if (in_t == FO_I4 && out_t == FO_I4) launch_pack_i4(rt->stream, out->ptr, (const int32_t*)O, (uint64_t)out_count);
  }
}

}  // namespace

extern "C" {

int32_t fo_contraction(fo_runtime* rt, fo_buffer* out, const fo_buffer* lhs, const fo_buffer* rhs, fo_dtype in_t,
                       fo_dtype out_t, const char* lhs_map, const char* rhs_map, const char* pre_reduce,
                       const char* out_map) {
  return guard([&] {
    contraction_impl(rt, out, lhs, rhs, in_t, out_t, lhs_map, rhs_map, pre_reduce, out_map, false);
  });
}

int32_t fo_contraction_noalloc(fo_runtime* rt, fo_buffer* out, const fo_buffer* lhs, const fo_buffer* rhs,
                               fo_dtype in_t, fo_dtype out_t, const char* lhs_map, const char* rhs_map,
                               const char* pre_reduce, const char* out_map) {
  return guard([&] {
    contraction_impl(rt, out, lhs, rhs, in_t, out_t, lhs_map, rhs_map, pre_reduce, out_map, true);
  });
}

// ---- fused chains ----------------------------------------------------------------------------------

int32_t fo_rmsnorm_softmax(fo_runtime* rt, fo_buffer* out, const fo_buffer* x, const fo_buffer* gain, int64_t rows,
                           int64_t cols, float eps) {
  return guard([&] {
    check_rt(rt);
    check_buf(out, "out");
    note_write(out);
    check_buf(x, "x");
    check_buf(gain, "gain");
    require(rows > 0 && cols > 0, "rmsnorm_softmax: empty shape");
    require((uint64_t)(rows * cols * 2) <= x->bytes && (uint64_t)(rows * cols * 2) <= out->bytes &&
                (uint64_t)(cols * 2) <= gain->bytes,
            "rmsnorm_softmax: shape exceeds a buffer");
    set_device(rt);
    TraceScope trace_span(rt, "rmsnorm_softmax");
    launch_rmsnorm_softmax(rt->stream, (uint16_t*)out->ptr, (const uint16_t*)x->ptr, (const uint16_t*)gain->ptr, rows,
                           cols, eps);
  });
}

int32_t fo_attention_prefill(fo_runtime* rt, fo_buffer* out, const fo_buffer* q, const fo_buffer* k,
                             const fo_buffer* v, int64_t batch, int64_t heads, int64_t seq, int64_t head_dim,
                             float sqrt_d, int32_t causal, const fo_buffer* row_max) {
  return guard([&] {
    check_rt(rt);
    check_buf(out, "out");
    note_write(out);
    check_buf(q, "q");
    check_buf(k, "k");
    check_buf(v, "v");
    require(batch > 0 && heads > 0 && seq > 0, "attention: empty shape");
    require(head_dim == 64 || head_dim == 128, "attention: head_dim must be 64 or 128");
    uint64_t bytes = (uint64_t)(batch * heads * seq * head_dim * 2);
    require(bytes <= q->bytes && bytes <= k->bytes && bytes <= v->bytes && bytes <= out->bytes,
            "attention: shape exceeds a buffer");
    if (row_max) {
      check_buf(row_max, "row_max");
      require((uint64_t)(batch * heads * seq) * 4 <= row_max->bytes, "attention: row_max smaller than batch*heads*seq");
      require((uintptr_t)row_max->ptr % 4 == 0, "attention: row_max not aligned");
    }
    set_device(rt);
    TraceScope trace_span(rt, "attention_prefill");
    launch_attention_prefill(rt->stream, (uint16_t*)out->ptr, (const uint16_t*)q->ptr, (const uint16_t*)k->ptr,
                             (const uint16_t*)v->ptr, row_max ? (const float*)row_max->ptr : nullptr, batch, heads,
                             seq, head_dim, sqrt_d, causal);
  });
}

int32_t fo_gemm_w8a8_dequant(fo_runtime* rt, fo_buffer* out, fo_buffer* acc_out, const fo_buffer* a,
                             const fo_buffer* w, const fo_buffer* scale, int64_t m, int64_t n, int64_t k) {
  return guard([&] {
    check_rt(rt);
    check_buf(out, "out");
    note_write(out);
    note_write(acc_out);
    check_buf(a, "a");
    check_buf(w, "w");
    check_buf(scale, "scale");
    require(m > 0 && n > 0 && k > 0, "w8a8: empty shape");
    require((uint64_t)(m * k) <= a->bytes && (uint64_t)(n * k) <= w->bytes && (uint64_t)(n * 4) <= scale->bytes &&
                (uint64_t)(m * n * 2) <= out->bytes,
            "w8a8: shape exceeds a buffer");
    if (acc_out) {
      check_buf(acc_out, "acc_out");
      require((uint64_t)(m * n * 4) <= acc_out->bytes, "w8a8: shape exceeds acc_out");
    }
    set_device(rt);
    TraceScope trace_span(rt, "gemm_w8a8_dequant");
    launch_w8a8(rt->stream, (uint16_t*)out->ptr, acc_out ? (int32_t*)acc_out->ptr : nullptr, (const int8_t*)a->ptr,
                (const int8_t*)w->ptr, (const float*)scale->ptr, m, n, k, rt->gemm_ws);
  });
}

int32_t fo_mlp(fo_runtime* rt, fo_buffer* pred_i32, fo_buffer* logits, const fo_buffer* x, const fo_buffer* w1,
               const fo_buffer* b1, const fo_buffer* w2, const fo_buffer* b2, int64_t batch, int64_t in_features,
               int64_t hidden, int64_t out_features) {
  return guard([&] {
    check_rt(rt);
    check_buf(pred_i32, "pred");
    note_write(pred_i32);
    note_write(logits);
    check_buf(x, "x");
    check_buf(w1, "w1");
    check_buf(b1, "b1");
    check_buf(w2, "w2");
    check_buf(b2, "b2");
    require(batch > 0 && in_features > 0 && hidden > 0 && out_features > 0, "mlp: empty shape");
    require(hidden <= 1024 && out_features <= 64, "mlp: hidden <= 1024 and out_features <= 64");
    require((uint64_t)(batch * in_features * 2) <= x->bytes && (uint64_t)(hidden * in_features * 2) <= w1->bytes &&
                (uint64_t)(hidden * 2) <= b1->bytes && (uint64_t)(out_features * hidden * 2) <= w2->bytes &&
                (uint64_t)(out_features * 2) <= b2->bytes && (uint64_t)(batch * 4) <= pred_i32->bytes,
            "mlp: shape exceeds a buffer");
    if (logits) {
      check_buf(logits, "logits");
      require((uint64_t)(batch * out_features * 2) <= logits->bytes, "mlp: shape exceeds logits");
    }
    set_device(rt);
    TraceScope trace_span(rt, "mlp");
    launch_mlp(rt->stream, (int32_t*)pred_i32->ptr, logits ? (uint16_t*)logits->ptr : nullptr,
               (const uint16_t*)x->ptr, (const uint16_t*)w1->ptr, (const uint16_t*)b1->ptr, (const uint16_t*)w2->ptr,
               (const uint16_t*)b2->ptr, batch, in_features, hidden, out_features);
  });
}

// ---- safetensors ----------------------------------------------------------------------------------

int32_t fo_safetensors_info(const char* path, const char* name, int32_t* dtype, int64_t* shape, int32_t cap,
                            int32_t* rank, uint64_t* data_begin, uint64_t* data_end) {
  return guard([&] {
    require(path != nullptr && name != nullptr, "safetensors: path or name is NULL");
    File file(path);
    TensorInfo info = find_tensor(file, path, name);
    if (dtype) *dtype = dtype_code(info.dtype);
    if (rank) *rank = (int32_t)info.shape.size();
    for (int32_t i = 0; shape && i < cap && i < (int32_t)info.shape.size(); ++i) shape[i] = info.shape[i];
    if (data_begin) *data_begin = info.begin;
    if (data_end) *data_end = info.end;
  });
}

int32_t fo_safetensors_load(fo_runtime* rt, fo_buffer* dst, const char* path, const char* name, fo_dtype t,
                            const char* element_map) {
  return guard([&] {
    check_rt(rt);
    not_recording(rt, "fo_safetensors_load");
    check_buf(dst, "dst");
    note_write(dst);
    require(path != nullptr && name != nullptr && element_map != nullptr, "safetensors: NULL argument");
    fm::NodeP m = fm::parse_json(element_map);
    File file(path);
    TensorInfo info = find_tensor(file, path, name);
    std::vector<int64_t> want;
    flat_shape(m, want);
    // TensorInvalidInfo (memory.rs:213-220): the shape and the byte length must match the mapping.
    require(info.shape == want, "safetensors: the tensor's shape is not the element mapping's pair-flattened sizes");
    const uint64_t bytes = span_bytes(t, (uint64_t)fm::size(m));
    require(info.end - info.begin == bytes, "safetensors: the tensor's byte length does not match the mapping");
    require(bytes <= dst->bytes, "safetensors: dst buffer smaller than the tensor");
    set_device(rt);
    TraceScope trace_span(rt, "safetensors_load");
    // Stream through a pinned staging buffer in 64 MiB pieces.
    const uint64_t piece = std::min<uint64_t>(bytes, 64ull << 20);
    if (bytes == 0) return;
    void* stage = nullptr;
    FO_HIP(hipHostMalloc(&stage, piece, hipHostMallocDefault));
    std::unique_ptr<void, void (*)(void*)> guard_stage(stage, [](void* p) { (void)hipHostFree(p); });
    std::fseek(file.f, (long)info.begin, SEEK_SET);
    for (uint64_t done = 0; done < bytes; done += piece) {
      const uint64_t len = std::min(piece, bytes - done);
      require(std::fread(stage, 1, len, file.f) == len, "safetensors: short read");
      FO_HIP(hipMemcpyAsync((uint8_t*)dst->ptr + done, stage, len, hipMemcpyHostToDevice, rt->stream));
      FO_HIP(hipStreamSynchronize(rt->stream));
    }
  });
}

}  // extern "C"
