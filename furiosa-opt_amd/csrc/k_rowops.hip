// Fused vector-engine row chain: RMSNorm then row softmax, one HBM pass (read x, write out).
// Rounding points follow the reference RMSNorm kernel (furiosa-opt-examples/src/transformer/
// kernel/rmsnorm.rs:9-78): fetch_cast bf16 -> f32; x*x (MulF with the stash) summed by the intra-
// slice reduce; fp_div by the column count; clip Add eps; Sqrt; (x * g) / r in f32; cast to bf16 at
// commit. The softmax re-fetches the committed bf16 values: max, exp(y - max), sum, divide, cast.
//
// Layout: a lane holds 16-byte chunks of its row (8 bf16 each), consecutive lanes consecutive chunks, so a
// wave's load or store is 1 KiB contiguous. exp(y - max) is held in f32 registers from the sum to the
// output, so each element is read, exponentiated and written once. Two kernels:
//   * k_rmsnorm_softmax_row (up to 32768 columns, any row length): one to sixteen waves per row;
//   * k_rmsnorm_softmax_dma (2048 or 4096 columns, many rows): one wave per row, persistent waves, the next row
//     fetched into LDS by DMA while the current one is computed, the gain staged once per block.
// Bound by HBM when large (5.1-5.4 TB/s, what a large copy reaches) and by the launch and one memory
// round trip when small.
//
// Numerics. This file is compiled with f32 denormals flushed (inputs and results, sign kept),
// which is the reference's own numeric model: its bf16 widen and narrow flush every subnormal to a
// signed zero (float/bf16.rs:16-40). With that mode a bf16 -> f32 widen is a plain shift (a
// subnormal reads as zero in every later op), a subnormal result flushes before the narrow, and
// the narrow is the hardware round-to-nearest-even v_cvt_pk_bf16_f32. The one case left is a
// non-finite value (NaN payloads and inf - inf), which the reference canonicalises: a row whose
// sum of squares is non-finite, whose mean square may not be positive (a division by zero) or whose gain
// reaches kGainMax is computed by the exact per-element path.
//   * (x*g)/r is the correctly rounded quotient q' = RN(q + e*y), q = RN(a*y), e = a - q*r (exact,
//     one FMA), y = RN(1/r) (Markstein's correction, exact for normal operands and results);
//   * exp and the final division feed only the output's bf16 narrow, so they use the hardware exp2
//     and reciprocal (<= 2 f32 ulps; a flip of the narrow from them is a 1-ulp change);
//   * the row max is taken on f32 y: rounding to nearest is monotone, so bf16(max y) = max bf16(y).
#include <hip/hip_runtime.h>

#include "launch_rules.hpp"
#include "runtime.hpp"

namespace fo {
namespace {

typedef __attribute__((__vector_size__(4 * sizeof(int)))) int i32x4_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2_t;
typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2_t;

// Wave64 reductions to a uniform value: four DPP steps combine the 16 lanes of each row (swap
// neighbours, swap pairs, mirror within 8, mirror within 16; after each step the lanes of a group
// hold equal values), then the four row results are read out with v_readlane. DPP moves data
// between lanes inside the VALU, without the LDS round trip of ds_bpermute. All 64 lanes must be
// active.
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
constexpr int kDppXor1 = 0xb1;         // quad_perm [1, 0, 3, 2]
constexpr int kDppXor2 = 0x4e;         // quad_perm [2, 3, 0, 1]
constexpr int kDppHalfMirror = 0x141;  // row_half_mirror
constexpr int kDppMirror = 0x140;      // row_mirror
__device__ __forceinline__ float lane_f(float v, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}
__device__ __forceinline__ float wave_sum(float v) {
  v += dpp<kDppXor1>(v);
  v += dpp<kDppXor2>(v);
  v += dpp<kDppHalfMirror>(v);
  v += dpp<kDppMirror>(v);
  return (lane_f(v, 0) + lane_f(v, 16)) + (lane_f(v, 32) + lane_f(v, 48));
}
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, dpp<kDppXor1>(v));
  v = fmaxf(v, dpp<kDppXor2>(v));
  v = fmaxf(v, dpp<kDppHalfMirror>(v));
  v = fmaxf(v, dpp<kDppMirror>(v));
  return fmaxf(fmaxf(lane_f(v, 0), lane_f(v, 16)), fmaxf(lane_f(v, 32), lane_f(v, 48)));
}

// A pointer the compiler cannot prove wave-uniform but is by construction (so a buffer descriptor
// built from it stays in SGPRs).
__device__ __forceinline__ const void* uniform_ptr(const void* p) {
  uint64_t v = (uint64_t)p;
  uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (const void*)(((uint64_t)hi << 32) | lo);
}

// a.lo * b.lo + a.hi * b.hi + c on packed bf16 pairs (v_dot2_f32_bf16).
__device__ __forceinline__ float dot2_bf16(int a, int b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, a), __builtin_bit_cast(bf16x2_t, b), c, false);
}

// Plain widen of the low / high bf16 of a packed word (subnormals read as zero in flush mode).
__device__ __forceinline__ float lo_raw(uint32_t w) { return bits_f32(w << 16); }
__device__ __forceinline__ float hi_raw(uint32_t w) { return bits_f32(w & 0xffff0000u); }

// Round two f32 to packed bf16 with the hardware RNE convert.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  f32x2_t v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// With gains below this, and a finite sum of squares, |y_i| <= sqrt(cols) * max|g| < 2^7.5 * 2^21 at the
// 32768 columns the kernels take (|x_i| <= sqrt(ss), r >= sqrt(ss / cols)). exp2 of the fused
// y * log2(e) - RN(max * log2(e)) leaves the rounding of the product, up to 2^-24 of it, as a common
// factor of the row: below 2^6 in the exponent then, which the sum divides out; past it the row's
// exponentials overflow or all vanish.
constexpr float kGainMax = 0x1p21f;

// The exact per-element path (reference rules at every rounding point), for rows holding a
// non-finite value. Reads the row again from global memory.
__device__ void row_exact(uint16_t* __restrict__ orow, const uint16_t* __restrict__ xr,
                          const uint16_t* __restrict__ gain, int cols, float eps, int lane) {
  float ss = 0.f;
  for (int i = lane; i < cols; i += 64) {
    float f = bf16_to_f32(xr[i]);
    ss = __fadd_rn(ss, __fmul_rn(f, f));
  }
  ss = wave_sum(ss);
  float r = sqrt_rn(__fadd_rn(__fdiv_rn(ss, (float)cols), eps));
  float mx = -INFINITY;
  for (int i = lane; i < cols; i += 64) {
    float y = bf16_to_f32(f32_to_bf16(__fdiv_rn(__fmul_rn(bf16_to_f32(xr[i]), bf16_to_f32(gain[i])), r)));
    mx = fmaxf(mx, y);
  }
  mx = wave_max(mx);
  float s = 0.f;
  for (int i = lane; i < cols; i += 64) {
    float y = bf16_to_f32(f32_to_bf16(__fdiv_rn(__fmul_rn(bf16_to_f32(xr[i]), bf16_to_f32(gain[i])), r)));
    s += expf(__fsub_rn(y, mx));
  }
  s = wave_sum(s);
  for (int i = lane; i < cols; i += 64) {
    float y = bf16_to_f32(f32_to_bf16(__fdiv_rn(__fmul_rn(bf16_to_f32(xr[i]), bf16_to_f32(gain[i])), r)));
    orow[i] = f32_to_bf16(__fdiv_rn(expf(__fsub_rn(y, mx)), s));
  }
}

// Rows of 2048 or 4096 columns: one wave per row, persistent waves, the next row fetched into LDS
// by DMA (buffer_load ... lds) while the current one is computed. A register prefetch would not
// stay in flight: with this row's stores also outstanding the compiler waits for every access
// before touching the prefetched registers. Here the only wait on vector memory is explicit and
// sits just before the row's stores, when the DMA issued at the start of the row and the previous
// row's stores are a whole row's compute old. exp(y - max) is kept in registers from the sum to
// the output, so each element is exponentiated once.
typedef __attribute__((address_space(3))) void* lds_ptr_t;
// The row streams through once: the DMA reads carry the sc0 and nt cache-policy bits (1.2% faster
// on the 8192 x 4096 config than default caching).
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rsrc, void* lds, uint32_t voff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)lds, 16, voff, 0, 0, 3);
#endif
}
constexpr int waitcnt_vm0 = (0 & 15) | (7 << 4) | (15 << 8);  // vmcnt(0); lgkmcnt, expcnt left alone
constexpr int waitcnt_lgkm0 = 15 | (7 << 4) | (0 << 8) | (3 << 14);  // lgkmcnt(0); vmcnt left alone

// Waves per block, sharing the staged gain: one block of sixteen fills a CU (144 KiB of LDS). Two
// blocks of eight per CU measured 4% slower on the 8192 x 4096 config.
constexpr int kDmaWaves = 16;
template <int NCH>
__global__ void __launch_bounds__(64 * kDmaWaves) k_rmsnorm_softmax_dma(uint16_t* __restrict__ out, const uint16_t* __restrict__ x,
                                                             const uint16_t* __restrict__ gain, int64_t rows,
                                                             float cols_f, float eps) {
  constexpr int cols = NCH * 512;
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const int64_t wave = (int64_t)blockIdx.x * kDmaWaves + wv;
  const int64_t nwaves = (int64_t)gridDim.x * kDmaWaves;
  __shared__ __attribute__((aligned(16))) float sg[cols];
  __shared__ __attribute__((aligned(16))) i32x4_t sx[kDmaWaves][NCH * 64];  // the wave's next row: chunk c at [c * 64 + lane]
  // Chunk c of a row (1 KiB) lands at sx[wv][c * 64]: lane l's 16 bytes at + 16 l, where lane l reads
  // them back (conflict-free b128 reads).
  auto fetch = [&](int64_t r) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void*>(uniform_ptr(x + r * cols)), (short)0, cols * 2, 0x00020000);
#pragma unroll
    for (int c = 0; c < NCH; ++c) dma16(rs, &sx[wv][c * 64], (uint32_t)(c * 1024 + lane * 16));
  };
  int64_t row = __builtin_amdgcn_readfirstlane((int)wave);
  if (row < rows) fetch(row);  // overlaps the gain staging below
  // The gain row is shared by every row: widen it once per block into LDS (reference widen rule),
  // and note whether it holds a non-finite value or a magnitude of kGainMax or more.
  // Each thread checks the gain values it stages; one workgroup reduction combines the checks (it
  // also orders the staging before every wave's reads).
  int bad_local = 0;
  for (int i = threadIdx.x; i < cols; i += blockDim.x) {
    const float gv = bf16_to_f32(gain[i]);
    sg[i] = gv;
    bad_local |= !(__builtin_fabsf(gv) < kGainMax);
  }
  __syncthreads();
  const bool gain_bad = __syncthreads_or(bad_local) != 0;
  if (row >= rows) return;
  // Sums of squares from here on have a positive mean square: with an eps every one, without it those that the
  // division can't flush. Comparing the sum itself keeps the division off the branch (8000 x 2048: 13.6 us with it).
  const float ss_min = gain_bad ? INFINITY : eps >= 0x1p-126f ? 0.f : eps >= 0.f ? 0x1p-100f : INFINITY;
  __builtin_amdgcn_s_waitcnt(waitcnt_vm0);

  for (; row < rows; row += nwaves) {
    i32x4_t v[NCH];
    __asm__ volatile("" ::: "memory");
#pragma unroll
    for (int c = 0; c < NCH; ++c) v[c] = sx[wv][c * 64 + lane];
    __builtin_amdgcn_s_waitcnt(waitcnt_lgkm0);  // the row is in registers before its buffer is refilled
    __asm__ volatile("" ::: "memory");
    if (row + nwaves < rows) fetch(row + nwaves);
    // Sum of squares by v_dot2_f32_bf16 on the packed pairs (two chains). The reference rounds each
    // square and then each partial sum; the squares of bf16 values are exact in f32, and its
    // reduction order is not this one anyway, so the sums agree to f32 rounding.
    float ss0 = 0.f, ss1 = 0.f;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      ss0 = dot2_bf16(v[c][0], v[c][0], ss0);
      ss1 = dot2_bf16(v[c][1], v[c][1], ss1);
      ss0 = dot2_bf16(v[c][2], v[c][2], ss0);
      ss1 = dot2_bf16(v[c][3], v[c][3], ss1);
    }
    const float ss = wave_sum(ss0 + ss1);
    uint16_t* orow = out + row * cols;
    if (!(ss >= ss_min && ss < INFINITY)) {
      row_exact(orow, x + row * cols, gain, cols, eps, lane);
      __builtin_amdgcn_s_waitcnt(waitcnt_vm0);
      continue;
    }
    const float ms = __fadd_rn(__fdiv_rn(ss, cols_f), eps);  // fp_div, then clip Add eps
    const float r = sqrt_rn(ms);                              // FpUnaryOp::Sqrt
    const float rinv = __fdiv_rn(1.0f, r);
    // y = bf16((x * g) / r), kept packed; row max on the f32 values
    float mx0 = -INFINITY, mx1 = -INFINITY;  // two chains of three-way maxima
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      f32x4_t g0 = *(const f32x4_t*)(sg + (c * 64 + lane) * 8);
      f32x4_t g1 = *(const f32x4_t*)(sg + (c * 64 + lane) * 8 + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t u = (uint32_t)v[c][e];
        float glo = e < 2 ? g0[2 * e] : g1[2 * e - 4];
        float ghi = e < 2 ? g0[2 * e + 1] : g1[2 * e - 3];
        float ylo = div_cr(lo_raw(u) * glo, r, rinv);
        float yhi = div_cr(hi_raw(u) * ghi, r, rinv);
        if (e & 1)
          mx1 = fmaxf(fmaxf(mx1, ylo), yhi);
        else
          mx0 = fmaxf(fmaxf(mx0, ylo), yhi);
        v[c][e] = (int)pack_bf16(ylo, yhi);
      }
    }
    float mx = wave_max(fmaxf(mx0, mx1));
    mx = bits_f32(pack_bf16(mx, mx) << 16);  // the max of the committed bf16 values
    // softmax: e = exp(y - max) kept in f32, s = sum(e), out = bf16(e / s)
    const float L2E = 1.4426950408889634f;
    const float mxl = mx * L2E;
    float ex[NCH][8];
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < NCH; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t u = (uint32_t)v[c][e];
        ex[c][2 * e] = __builtin_amdgcn_exp2f(__builtin_fmaf(lo_raw(u), L2E, -mxl));
        ex[c][2 * e + 1] = __builtin_amdgcn_exp2f(__builtin_fmaf(hi_raw(u), L2E, -mxl));
        s += ex[c][2 * e];
        s += ex[c][2 * e + 1];
      }
    s = wave_sum(s);
    const float sinv = __builtin_amdgcn_rcpf(s);
    // The next row's DMA and the previous row's stores are complete before these stores go out, so
    // no vector memory access is pending at the next row's LDS reads.
    __builtin_amdgcn_s_waitcnt(waitcnt_vm0);
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      i32x4_t o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (int)pack_bf16(ex[c][2 * e] * sinv, ex[c][2 * e + 1] * sinv);
      __builtin_nontemporal_store(o, (i32x4_t*)(orow + (c * 64 + lane) * 8));
    }
  }
}

template <int NCH>
void rs_dma_launch(hipStream_t s, uint16_t* out, const uint16_t* x, const uint16_t* g, int64_t rows, float eps) {
  static int64_t resident_blocks = [] {
    int dev = 0, per_cu = 1, cus = 1;
    (void)hipGetDevice(&dev);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_rmsnorm_softmax_dma<NCH>, 64 * kDmaWaves, 0) != hipSuccess ||
        per_cu < 1)
      per_cu = 1;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) cus = 256;
    return (int64_t)per_cu * cus;
  }();
  int64_t blocks = (rows + kDmaWaves - 1) / kDmaWaves;
  if (blocks > resident_blocks) blocks = resident_blocks;
  hipLaunchKernelGGL(k_rmsnorm_softmax_dma<NCH>, dim3((unsigned)blocks), dim3(64 * kDmaWaves), 0, s, out, x, g, rows,
                     (float)(NCH * 512), eps);
}

// A row of up to 32768 columns over W waves, P elements a lane held in registers from the load to the
// output (x, then y, then exp(y - max)), so the row is read once. Element e of chunk c of thread t is
// column (c * T + t) * 8 + e, T = 64 W. Chunks are 16-byte accesses at any even address (rows of an
// odd length start anywhere); the row's last, partial chunk goes element by element. The gain is read
// per row, from the caches.
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
typedef u16x8 u16x8_any __attribute__((aligned(2)));

template <int P, int W, bool NT>
__global__ void __launch_bounds__(W < 4 ? 256 : 64 * W) k_rmsnorm_softmax_row(uint16_t* __restrict__ out,
                                                                         const uint16_t* __restrict__ x,
                                                                         const uint16_t* __restrict__ gain, int64_t rows,
                                                                         int cols, float eps) {
  constexpr int NC = P / 8;
  constexpr int T = 64 * W;
  constexpr int R = W < 4 ? 4 / W : 1;  // rows per block
  const int lane = threadIdx.x & 63;
  const int wave = (threadIdx.x >> 6) % W, slot = (threadIdx.x >> 6) / W;
  const int64_t row = (int64_t)blockIdx.x * R + slot;
  const bool live = row < rows;  // no early return: the barriers below are the block's
  const int t = wave * 64 + lane;
  __shared__ float red[3][R][W];
  auto combine = [&](int k, float v, bool max) __attribute__((always_inline)) {
    v = max ? wave_max(v) : wave_sum(v);
    if (W > 1) {
      if (lane == 0) red[k][slot][wave] = v;
      __syncthreads();
      v = red[k][slot][0];
#pragma unroll
      for (int i = 1; i < W; ++i) v = max ? fmaxf(v, red[k][slot][i]) : v + red[k][slot][i];
    }
    return v;
  };
  const uint16_t* xr = x + row * cols;
  uint16_t* orow = out + row * cols;
  u16x8 xv[NC], gv[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int j = (c * T + t) * 8;
    xv[c] = gv[c] = (u16x8)(uint16_t)0;
    const bool all = (c + 1) * T * 8 <= cols;  // uniform: no lane of the row needs a check
    if (live && (all || j + 8 <= cols)) {
      xv[c] = NT ? __builtin_nontemporal_load((const u16x8_any*)(xr + j)) : *(const u16x8_any*)(xr + j);
      gv[c] = *(const u16x8_any*)(gain + j);
    } else if (live && j < cols) {
#pragma unroll
      for (int e = 0; e < 7; ++e)
        if (j + e < cols) {
          xv[c][e] = xr[j + e];
          gv[c][e] = gain[j + e];
        }
    }
  }
  float y[P];
  float ss = 0.f;
  bool bad = false;  // a gain of kGainMax or more
#pragma unroll
  for (int i = 0; i < P; ++i) {
    y[i] = bits_f32((uint32_t)xv[i / 8][i % 8] << 16);
    ss = __builtin_fmaf(y[i], y[i], ss);  // a bf16 square is exact in f32
    bad |= !(__builtin_fabsf(bits_f32((uint32_t)gv[i / 8][i % 8] << 16)) < kGainMax);
  }
  ss = combine(0, bad ? INFINITY : ss, false);
  const float ms = __fadd_rn(__fdiv_rn(ss, (float)cols), eps);  // fp_div, then clip Add eps
  const bool exact = !__builtin_isfinite(ss) || !(ms > 0.f);  // uniform over the row's waves
  const float r = sqrt_rn(ms);                                    // FpUnaryOp::Sqrt
  const float rinv = __fdiv_rn(1.0f, r);
  float mx = -INFINITY;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int past = cols - (c * T + t) * 8;  // elements of the chunk inside the row
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      float* v = y + c * 8 + i;
#pragma unroll
      for (int e = 0; e < 2; ++e) v[e] = div_cr(v[e] * bits_f32((uint32_t)gv[c][i + e] << 16), r, rinv);
      const uint32_t u = pack_bf16(v[0], v[1]);
      v[0] = lo_raw(u);
      v[1] = hi_raw(u);
    }
    if ((c + 1) * T * 8 > cols) {  // uniform
#pragma unroll
      for (int i = 0; i < 8; ++i) y[c * 8 + i] = i < past ? y[c * 8 + i] : -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < 8; i += 2) mx = fmaxf(fmaxf(mx, y[c * 8 + i]), y[c * 8 + i + 1]);
  }
  mx = combine(1, mx, true);
  const float L2E = 1.4426950408889634f;
  const float mxl = mx * L2E;
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < P; ++i) {
    y[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(y[i], L2E, -mxl));
    s += y[i];
  }
  s = combine(2, s, false);
  if (!live) return;
  if (exact) {
    if (wave == 0) row_exact(orow, xr, gain, cols, eps, lane);
    return;
  }
  const float sinv = __builtin_amdgcn_rcpf(s);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int j = (c * T + t) * 8;
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = pack_bf16(y[c * 8 + 2 * e] * sinv, y[c * 8 + 2 * e + 1] * sinv);
    const u16x8 o = __builtin_bit_cast(u16x8, w);
    const bool all = (c + 1) * T * 8 <= cols;
    if (all || j + 8 <= cols) {
      if (NT)
        __builtin_nontemporal_store(o, (u16x8_any*)(orow + j));
      else
        *(u16x8_any*)(orow + j) = o;
    } else if (j < cols) {
#pragma unroll
      for (int e = 0; e < 7; ++e)
        if (j + e < cols) orow[j + e] = o[e];
    }
  }
}

template <int P, int W>
void rs_row_launch(hipStream_t s, uint16_t* out, const uint16_t* x, const uint16_t* g, int64_t rows, int64_t cols,
                   float eps, bool stream) {
  constexpr int R = W < 4 ? 4 / W : 1;
  for_row_pieces(rows, 64 * W, [&](int64_t first, int64_t n) {
    const dim3 grid((unsigned)((n + R - 1) / R)), block(W < 4 ? 256 : 64 * W);
    uint16_t* o = out + first * cols;
    const uint16_t* in = x + first * cols;
    if (stream)
      hipLaunchKernelGGL((k_rmsnorm_softmax_row<P, W, true>), grid, block, 0, s, o, in, g, n, (int)cols, eps);
    else
      hipLaunchKernelGGL((k_rmsnorm_softmax_row<P, W, false>), grid, block, 0, s, o, in, g, n, (int)cols, eps);
  });
}

// Rows past 32768 columns: the exact per-element path, one wave per row.
__global__ void __launch_bounds__(256) k_rmsnorm_softmax_any(uint16_t* __restrict__ out, const uint16_t* __restrict__ x,
                                                             const uint16_t* __restrict__ gain, int64_t rows, int64_t cols,
                                                             float eps) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  row_exact(out + row * cols, x + row * cols, gain, (int)cols, eps, lane);
}

}  // namespace

void launch_rmsnorm_softmax(hipStream_t s, uint16_t* out, const uint16_t* x, const uint16_t* gain, int64_t rows,
                            int64_t cols, float eps) {
  require((rows + 3) / 4 < (1ll << 31), "rmsnorm_softmax: too many rows");
  require(cols < (1ll << 30), "rmsnorm_softmax: too many columns");
  // Measured as the kernel alone in a recorded graph, us (one box; DMA is k_rmsnorm_softmax_dma, exact
  // the per-element path that took every column count the DMA form does not):
  //     rows, cols     row kernel   before        rows, cols     row kernel   before
  //     500, 512          3.1     4.4 (DMA)       500, 3072         4.5     41 (exact)
  //     32768, 1024      24.4    26.2 (DMA)
  //     500, 4096         4.5    12.2 (DMA)       4096, 8192       28.7     30.8 (rows split over 4 waves)
  // The DMA form is kept where it is the faster one (norm_dma). W and P are the best of one to sixteen waves a row; wider rows want more waves while the
  // result is small (2048 columns: 3.7 us with 4 waves against 3.9 with 2 at 500 rows; 32.4 against 26.2 at
  // 16384). Past 10 MiB a tensor the accesses stream past the caches (1500, 4096: 7.9 against 9.1 us;
  // at 4 MiB 5.3 against 4.5).
  const bool aligned = (((uintptr_t)x | (uintptr_t)out | (uintptr_t)gain) & 15) == 0;
  const bool stream = rows * cols * 2 >= (10ll << 20);
  if (aligned && norm_dma(rows, cols)) {
    cols == 4096 ? rs_dma_launch<8>(s, out, x, gain, rows, eps) : rs_dma_launch<4>(s, out, x, gain, rows, eps);
  } else if (cols <= 32768) {
    if (cols <= 512)
      rs_row_launch<8, 1>(s, out, x, gain, rows, cols, eps, stream);
    else if (cols <= 1024)
      rs_row_launch<16, 1>(s, out, x, gain, rows, cols, eps, stream);
    else if (cols <= 2048 && !stream)
      rs_row_launch<8, 4>(s, out, x, gain, rows, cols, eps, stream);
    else if (cols <= 2048)
      rs_row_launch<16, 2>(s, out, x, gain, rows, cols, eps, stream);
    else if (cols <= 3072 && stream)
      rs_row_launch<24, 2>(s, out, x, gain, rows, cols, eps, stream);
    else if (cols <= 4096)
      rs_row_launch<16, 4>(s, out, x, gain, rows, cols, eps, stream);
    else if (cols <= 8192)
      rs_row_launch<16, 8>(s, out, x, gain, rows, cols, eps, stream);
    else if (cols <= 16384)
      rs_row_launch<16, 16>(s, out, x, gain, rows, cols, eps, stream);
    else
      rs_row_launch<32, 16>(s, out, x, gain, rows, cols, eps, stream);
  } else {
    for_row_pieces(rows, 64, [&](int64_t first, int64_t n) {
      hipLaunchKernelGGL(k_rmsnorm_softmax_any, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, s, out + first * cols,
                         x + first * cols, gain, n, cols, eps);
    });
  }
  FO_HIP(hipGetLastError());
}

}  // namespace fo
