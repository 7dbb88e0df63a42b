"""Timed cases of the framework's main paths, each through the public binding (`furiosa_hip`).

A case is a dict: `kind` names the entry point, the other keys its sizes and types. `prepare` makes
what a program holds before the call (inputs resident on the device, output buffers, mappings, a
recorded graph), `run` is one pass, `exact` the same values in 64 bits by plain torch.

Device buffers of the library are opaque handles, so a pass returns `DeviceView`s: tensors that know
their shape and type and copy the buffer's contents only when something reads them.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "furiosa-opt_amd"))

import furiosa_hip as fh  # noqa: E402
import furiosa_hip.decode as fd  # noqa: E402

DEVICE = "cuda" if torch.cuda.is_available() else "cpu"
SQRT_D = {64: 8.0, 128: 11.313708}
NORM_EPS = 1e-6

# name -> (library type, torch type, integer type of the raw bits)
TYPES = {
    "bf16": (fh.BF16, torch.bfloat16, torch.int16),
    "f32": (fh.F32, torch.float32, torch.int32),
    "i8": (fh.I8, torch.int8, torch.int8),
    "i32": (fh.I32, torch.int32, torch.int32),
    "f8e4m3": (fh.F8E4M3, torch.float8_e4m3fn, torch.uint8),
}


def listed():
    return [
        # A large matrix product (the headline benchmark's shape).
        {"name": "gemm_4096", "kind": "gemm", "types": "bf16,bf16", "m": 4096, "n": 4096, "k": 4096},
        # A prompt chunk of 500 tokens through the decoder's up projection (1024 -> 3072).
        {"name": "gemm_chunk500", "kind": "gemm", "types": "bf16,bf16", "m": 500, "n": 3072, "k": 1024},
        # A ragged product whose rows don't start at 16-byte addresses, with the f32 result.
        {"name": "gemm_ragged", "kind": "gemm", "types": "bf16,f32", "m": 333, "n": 1000, "k": 777},
        # Quantized linear layer over a long prompt (the benchmark's shape) and over a decode batch.
        {"name": "w8a8_2048", "kind": "w8a8", "m": 2048, "n": 8192, "k": 8192},
        {"name": "w8a8_batch16", "kind": "w8a8", "m": 16, "n": 8192, "k": 8192},
        # Attention over a large prompt batch, and over one prompt of the decoder (16 heads of 128).
        {"name": "attention_2048", "kind": "attention", "batch": 4, "heads": 32, "seq": 2048, "dim": 128, "causal": True},
        {"name": "attention_600", "kind": "attention", "batch": 1, "heads": 16, "seq": 600, "dim": 128, "causal": True},
        # RMSNorm -> row softmax: the benchmark's shape, and a smaller one at the MLP's width.
        {"name": "norm_8192x4096", "kind": "norm", "rows": 8192, "cols": 4096},
        {"name": "norm_500x3072", "kind": "norm", "rows": 500, "cols": 3072},
        # The MNIST classifier on its batch of 64.
        {"name": "mlp_64", "kind": "mlp", "batch": 64, "inputs": 784, "hidden": 128, "outputs": 10},
        # A layout change of a ragged f32 matrix.
        {"name": "relayout_3000x1111", "kind": "relayout", "type": "f32", "a": 3000, "b": 1111, "c": 1, "dst": "B, A, C"},
        # One decoder layer for one token (projection, attention over two cache chunks, MLP),
        # recorded once as a graph and launched per token.
        {"name": "decode_layer_600", "kind": "decode", "pos": 600},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "w8a8", "w8a8", "attention", "attention", "norm", "norm", "mlp",
                       "relayout", "decode"])
    if kind == "gemm":
        types = rng.choice(["bf16,bf16", "bf16,bf16", "bf16,f32", "i8,i32", "f8e4m3,f32"])
        while True:
            m, n, k = _log(rng, 8, 4096), _log(rng, 64, 8192), _log(rng, 64, 8192)
            if m * n * k <= 4096 ** 3:
                break
        # Most contracted widths are whole 16-byte runs; the others are odd.
        if types == "f8e4m3,f32" or rng.random() < 0.75:
            k = max(64, k // 16 * 16)
        return {"kind": kind, "types": types, "m": m, "n": n, "k": k}
    if kind == "w8a8":
        return {"kind": kind, "m": _log(rng, 1, 2048), "n": _log(rng, 256, 8192), "k": _log(rng, 256, 8192) // 16 * 16}
    if kind == "attention":
        return {"kind": kind, "batch": rng.randint(1, 4), "heads": _log(rng, 1, 32), "seq": _log(rng, 16, 2048),
                "dim": rng.choice([64, 128]), "causal": rng.random() < 0.8}
    if kind == "norm":
        cols = 512 << rng.randint(0, 4) if rng.random() < 0.4 else _log(rng, 64, 8192)
        return {"kind": kind, "rows": _log(rng, 4, min(8192, 8192 * 4096 // cols)), "cols": cols}
    if kind == "mlp":
        return {"kind": kind, "batch": _log(rng, 1, 4096), "inputs": _log(rng, 64, 1024), "hidden": _log(rng, 16, 512),
                "outputs": rng.randint(2, 64)}
    if kind == "relayout":
        a, b, c = _log(rng, 16, 2048), _log(rng, 16, 2048), rng.choice([1, 1, 8, 64, 100])
        return {"kind": kind, "type": rng.choice(["f32", "bf16", "i8"]), "a": a, "b": b, "c": c,
                "dst": rng.choice(["B, A, C", "B, A, C", "C, A, B", "B, C, A"])}
    return {"kind": "decode", "pos": rng.randint(0, 4 * fd.T - 1)}


# ---- outputs -------------------------------------------------------------------------------------------


class DeviceView(torch.Tensor):
    """A library buffer as a tensor of a given type and shape; any torch operation on it reads the
    buffer first."""

    @staticmethod
    def __new__(cls, buf, dtype, shape):
        return torch.Tensor._make_wrapper_subclass(cls, shape, dtype=dtype, device=DEVICE)

    def __init__(self, buf, dtype, shape):
        self.buf, self.as_type, self.as_shape = buf, dtype, shape

    def contents(self):
        n = math.prod(self.as_shape)
        raw = self.buf.read(np.uint8, n * torch.empty(0, dtype=self.as_type).element_size())
        return torch.from_numpy(raw).to(DEVICE).view(self.as_type).reshape(self.as_shape)

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        def plain(x):
            if isinstance(x, cls):
                return x.contents()
            return type(x)(plain(y) for y in x) if isinstance(x, (list, tuple)) else x
        return func(*plain(args), **{k: plain(v) for k, v in (kwargs or {}).items()})


# ---- inputs --------------------------------------------------------------------------------------------


class _Process:
    runtime = None


def _rt():
    """The process's one runtime, as a program holds it."""
    if _Process.runtime is None:
        _Process.runtime = fh.Runtime(0)
    return _Process.runtime


def _inputs(case, seed):
    """The case's inputs as torch tensors, a function of the case and the seed alone."""
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed) * 7919 + 17)

    def normal(*shape, scale=1.0, loc=0.0):
        return (torch.randn(*shape, device=DEVICE, generator=gen) * scale + loc).to(torch.bfloat16)

    def uniform(*shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, device=DEVICE, generator=gen) * (hi - lo) + lo

    def whole(lo, hi, *shape):
        return torch.randint(lo, hi + 1, shape, device=DEVICE, generator=gen).to(torch.int8)

    kind = case["kind"]
    if kind == "gemm":
        t = TYPES[case["types"].split(",")[0]][1]
        make = (lambda *s: whole(-127, 127, *s)) if t == torch.int8 else (lambda *s: normal(*s).to(t))
        return dict(a=make(case["m"], case["k"]), b=make(case["n"], case["k"]))
    if kind == "w8a8":
        return dict(a=whole(-127, 127, case["m"], case["k"]), w=whole(-127, 127, case["n"], case["k"]),
                    scale=uniform(case["n"], lo=1e-3, hi=1e-2))
    if kind == "attention":
        shape = (case["batch"], case["heads"], case["seq"], case["dim"])
        return dict(q=normal(*shape), k=normal(*shape), v=normal(*shape))
    if kind == "norm":
        return dict(x=normal(case["rows"], case["cols"]), g=normal(case["cols"], scale=0.1, loc=1.0))
    if kind == "mlp":
        i, h, o = case["inputs"], case["hidden"], case["outputs"]
        return dict(x=uniform(case["batch"], i).to(torch.bfloat16), w1=normal(h, i, scale=0.05), b1=normal(h, scale=0.05),
                    w2=normal(o, h, scale=0.05), b2=normal(o, scale=0.05))
    if kind == "relayout":
        shape = (case["a"], case["b"], case["c"])
        if case["type"] == "i8":
            return dict(src=whole(-127, 127, *shape))
        return dict(src=normal(*shape).to(TYPES[case["type"]][1]))
    # decode: one layer's weights at the scale of trained ones, the residual stream, and the caches
    # holding the tokens before this one
    H, L, Q, P = fd.H, fd.L, fd.Q, fd.P
    got = dict(x=normal(H), q=normal(Q, H, scale=H ** -0.5), k=normal(P, H, scale=H ** -0.5),
               v=normal(P, H, scale=H ** -0.5), o=normal(H, Q, scale=Q ** -0.5), up=normal(L, H, scale=H ** -0.5),
               gate=normal(L, H, scale=H ** -0.5), down=normal(H, L, scale=L ** -0.5))
    for name, n in (("input_norm", H), ("post_norm", H), ("q_norm", fd.D), ("k_norm", fd.D)):
        got[name] = normal(n, scale=0.1, loc=1.0)
    chunks = case["pos"] // fd.T + 1
    for name in ("k_cache", "v_cache"):
        cache = normal(chunks * fd.T, fd.N, fd.D)
        cache[case["pos"]:] = 0
        got[name] = cache
    return got


def _up(t):
    """Uploads a tensor's bytes."""
    return _rt().upload(t.contiguous().view(torch.uint8).reshape(-1).cpu().numpy())


# ---- one pass ------------------------------------------------------------------------------------------


def prepare(case, seed):
    """{"call": one pass with no arguments, "out": its outputs, "keep": what the pass reads}."""
    rt, x, kind = _rt(), _inputs(case, seed), case["kind"]
    if kind == "decode":
        return _prepare_decode(case, x)
    dev = {name: _up(t) for name, t in x.items()}
    out = {}

    def output(name, type_name, *shape):
        t = TYPES[type_name][1]
        buf = rt.alloc(math.prod(shape) * torch.empty(0, dtype=t).element_size())
        out[name] = DeviceView(buf, t, shape)
        return buf

    if kind == "gemm":
        in_t, out_t = case["types"].split(",")
        s = dict(M=case["m"], N=case["n"], K=case["k"])
        maps = [fh.m(t, **s) for t in ("M, K", "N, K", "M, N, K", "M, N")]
        c = output("c", out_t, case["m"], case["n"])
        args = (c, dev["a"], dev["b"], TYPES[in_t][0], TYPES[out_t][0], *maps)
        call = lambda: rt.contraction(*args)  # noqa: E731
    elif kind == "w8a8":
        args = (output("out", "bf16", case["m"], case["n"]), None, dev["a"], dev["w"], dev["scale"], case["m"], case["n"],
                case["k"])
        call = lambda: rt.gemm_w8a8_dequant(*args)  # noqa: E731
    elif kind == "attention":
        b, h, s, d = (case[n] for n in ("batch", "heads", "seq", "dim"))
        args = (output("out", "bf16", b, h, s, d), dev["q"], dev["k"], dev["v"], b, h, s, d, SQRT_D[d], case["causal"])
        call = lambda: rt.attention_prefill(*args)  # noqa: E731
    elif kind == "norm":
        args = (output("out", "bf16", case["rows"], case["cols"]), dev["x"], dev["g"], case["rows"], case["cols"], NORM_EPS)
        call = lambda: rt.rmsnorm_softmax(*args)  # noqa: E731
    elif kind == "mlp":
        args = (output("pred", "i32", case["batch"]), output("logits", "bf16", case["batch"], case["outputs"]), dev["x"],
                dev["w1"], dev["b1"], dev["w2"], dev["b2"], case["batch"], case["inputs"], case["hidden"], case["outputs"])
        call = lambda: rt.mlp(*args)  # noqa: E731
    else:
        s = dict(A=case["a"], B=case["b"], C=case["c"])
        shape = tuple(s[n] for n in case["dst"].split(", "))
        dst = output("dst", case["type"], *shape)
        args = (dst, dev["src"], TYPES[case["type"]][0], fh.m("A, B, C", **s), fh.m(case["dst"], **s))

        def call():
            rt.transpose(*args)
            dst.flush()  # the next op reading dst would run the recorded relayout
    return {"call": call, "out": out, "keep": dev}


def _prepare_decode(case, x):
    """One layer recorded into a graph, as the pipeline records a token: weights, caches, masks and the
    token's inputs resident before the recording."""
    rt, T = _rt(), fd.T
    ops = fd.SeamOps(rt, fd.STEP_SIZES)
    chunk, row = divmod(case["pos"], T)
    dev = {name: _up(t) for name, t in x.items() if name not in ("k_cache", "v_cache")}
    caches = [tuple(_up(x[n][c * T:(c + 1) * T]) for n in ("k_cache", "v_cache")) for c in range(chunk + 1)]
    cos, sin = (ops.put(r) for r in fd.rope_row(case["pos"]))
    masks = [ops.put(np.ones(T, np.float32)) for _ in range(chunk)] + [ops.put(fd.causal_mask(row))]
    offset = ops.put(np.array([row * fd.ROW_STRIDE_ND], np.int32))
    rt.graph_begin()
    y = fd.layer_step(ops, dev["x"], dev, case["pos"], caches, cos, sin, masks=masks, offset=offset)
    graph = rt.graph_end()
    k, v = caches[chunk]
    out = dict(y=DeviceView(y, torch.bfloat16, (fd.H,)), k_cache=DeviceView(k, torch.bfloat16, (T, fd.N, fd.D)),
               v_cache=DeviceView(v, torch.bfloat16, (T, fd.N, fd.D)))
    return {"call": graph.launch, "out": out, "keep": (dev, caches, cos, sin, masks, offset, graph)}


def run(state):
    state["call"]()
    return state["out"]


# ---- what a pass cannot do without -----------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        ib, ob = (torch.empty(0, dtype=TYPES[t][1]).element_size() for t in case["types"].split(","))
        return {"bytes": (m * k + n * k) * ib + m * n * ob, "flops": 2 * m * n * k}
    if kind == "w8a8":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": m * k + n * k + 4 * n + 2 * m * n, "flops": 2 * m * n * k}
    if kind == "attention":
        heads, s, d = case["batch"] * case["heads"], case["seq"], case["dim"]
        pairs = s * (s + 1) // 2 if case["causal"] else s * s
        return {"bytes": 4 * heads * s * d * 2, "flops": 4 * heads * d * pairs}
    if kind == "norm":
        return {"bytes": 2 * case["rows"] * case["cols"] * 2 + 2 * case["cols"], "flops": 12 * case["rows"] * case["cols"]}
    if kind == "mlp":
        b, i, h, o = (case[n] for n in ("batch", "inputs", "hidden", "outputs"))
        return {"bytes": 2 * (b * i + h * i + h + o * h + o + b * o) + 4 * b, "flops": 2 * b * (i * h + h * o)}
    if kind == "relayout":
        n = case["a"] * case["b"] * case["c"]
        return {"bytes": 2 * n * torch.empty(0, dtype=TYPES[case["type"]][1]).element_size(), "flops": 0}
    weights = 2 * fd.H * fd.Q + 2 * fd.H * fd.P + 3 * fd.H * fd.L
    cached = (case["pos"] + 1) * 2 * fd.N * fd.D
    return {"bytes": 2 * (weights + cached + 2 * fd.H), "flops": 2 * weights + 2 * fd.G * cached}


def tolerance(case):
    kind = case["kind"]
    if kind == "relayout" or kind == "w8a8" or (kind == "gemm" and case["types"] == "i8,i32"):
        return "exact"  # moved bytes, whole numbers, and one rounding of an exact sum
    if kind == "gemm" and case["types"] == "bf16,f32":
        return {"rel": 5e-6, "max": 1e-4}  # 32-bit sums in another order
    if kind == "gemm" and case["types"] == "f8e4m3,f32":
        return {"rel": 2e-4, "max": 5e-3}  # the 8-bit matrix instruction sums at reduced precision
    if kind == "gemm":
        return {"rel": 1e-3, "max": 2e-2}  # one bf16 rounding of such sums: a few values move by one step
    if kind == "norm":
        return {"rel": 4e-3, "max": 4e-2}  # two bf16 roundings in sequence
    if kind == "attention":
        return {"rel": 1e-2, "max": 1e-1}  # weights rounded to bf16 at another scale, averages near zero
    if kind == "mlp":
        return {"rel": 1e-2, "max": 4e-2, "differ": 1e-2}  # four bf16 roundings; near ties of the argmax
    return {"rel": 1e-2, "max": 1e-1}  # a whole layer in bf16


# ---- 64-bit results ----------------------------------------------------------------------------------------


def exact(case, seed):
    x = {n: t.double() for n, t in _inputs(case, seed).items()}
    kind = case["kind"]
    if kind == "gemm":
        return dict(c=x["a"] @ x["b"].t().contiguous())
    if kind == "w8a8":
        return dict(out=(x["a"] @ x["w"].t().contiguous()) * x["scale"])
    if kind == "attention":
        s, d = case["seq"], case["dim"]
        hidden = torch.ones(s, s, dtype=torch.bool, device=DEVICE).triu(1) if case["causal"] else None
        q, k, v = (x[n].reshape(-1, s, d) for n in "qkv")
        out = torch.empty_like(q)
        for h in range(q.shape[0]):
            score = (q[h] @ k[h].t().contiguous()) / SQRT_D[d]
            if hidden is not None:
                score = score.masked_fill(hidden, -math.inf)
            out[h] = torch.softmax(score, 1) @ v[h]
        return dict(out=out.reshape(case["batch"], case["heads"], s, d))
    if kind == "norm":
        y = x["x"] * x["g"] / torch.sqrt((x["x"] ** 2).mean(1, keepdim=True) + NORM_EPS)
        return dict(out=torch.softmax(y, 1))
    if kind == "mlp":
        h = torch.relu(x["x"] @ x["w1"].t().contiguous() + x["b1"])
        return dict(pred=None, logits=h @ x["w2"].t().contiguous() + x["b2"])
    if kind == "relayout":
        return None  # moved bytes
    return _exact_decode(case, x)


def _exact_decode(case, x):
    """One decoder layer (RMSNorm, q/k/v with their head norms and RoPE, attention over the cached keys
    and this one, output projection, SiLU MLP, both residuals)."""
    pos, D, N, G = case["pos"], fd.D, fd.N, fd.G

    def norm(t, g):
        return t * g / torch.sqrt((t ** 2).mean(-1, keepdim=True) + fd.RMS_EPS)

    def bits(r):
        return torch.from_numpy(r.astype(np.int32) << 16).view(torch.float32).to(DEVICE).double()

    cos, sin = (bits(r) for r in fd.rope_row(pos))

    def rope(t):
        return t * cos + torch.cat([t[..., D // 2:], t[..., :D // 2]], -1) * sin

    y = norm(x["x"], x["input_norm"])
    q = rope(norm((x["q"] @ y).reshape(N, G, D), x["q_norm"]))
    x["k_cache"][pos] = rope(norm((x["k"] @ y).reshape(N, D), x["k_norm"]))
    x["v_cache"][pos] = (x["v"] @ y).reshape(N, D)
    keys, values = x["k_cache"][:pos + 1], x["v_cache"][:pos + 1]
    attended = [torch.softmax(q[n] @ keys[:, n].t().contiguous() / fd.SQRT_HEAD_DIM, 1) @ values[:, n].contiguous()
                for n in range(N)]
    x1 = x["x"] + x["o"] @ torch.stack(attended).reshape(-1)
    y = norm(x1, x["post_norm"])
    gate = x["gate"] @ y
    y = x1 + x["down"] @ ((x["up"] @ y) * gate * torch.sigmoid(gate))
    chunk = slice(pos // fd.T * fd.T, (pos // fd.T + 1) * fd.T)
    return dict(y=y, k_cache=x["k_cache"][chunk], v_cache=x["v_cache"][chunk])
