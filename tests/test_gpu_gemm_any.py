"""MFMA contractions whose operand rows start at any element address or whose K is not whole 16-byte chunks
(k_gemm staged through registers): small-integer operands, exact sums, compared bit for bit."""
import numpy as np
import pytest

import furiosa_hip as fh
from oracle import emulator as emu
from test_gpu_gemm_tiles import TYPES, narrowed, operands, product

pytestmark = pytest.mark.gpu

# K below a chunk (small outputs of it go to the vector-unit fold, 1000 x 777 x 2 to the tiles), around a stage
# (64 bf16, 128 i8), prefetch depths, shared tiles with an uneven last run, and the larger tile; rows past the last tile.
SIZES = [(8, 8, 1), (8, 9, 7), (65, 64, 63), (64, 65, 65), (70, 33, 127), (33, 70, 129), (64, 64, 255), (9, 100, 321),
         (40, 24, 6145), (128, 200, 3331), (333, 1000, 777), (2113, 1100, 71), (1500, 2000, 131),
         # either side of the shortest K that the tiles take
         (8, 8, 21), (9, 8, 49), (70, 33, 9), (70, 33, 33), (530, 530, 15), (530, 530, 17), (1000, 777, 2)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("types", ["bf16", "bf16-f32", "i8", "i8-i32"])
def test_gemm_any_alignment_exact(rt, size, types):
    m, n, k = size
    in_t, out_t = TYPES[types]
    rng = np.random.default_rng(m + n + k)
    av, a = operands(rng, in_t, m, k)
    bv, b = operands(rng, in_t, n, k)
    want = narrowed(product(av, bv), out_t)
    maps = [fh.m(t, M=m, N=n, K=k) for t in ("M, K", "N, K", "M, N, K", "M, N")]
    out = rt.upload(np.full(m * n, 0x5A, dtype=fh.NP_DTYPE[out_t]))
    print(f"gemm any {size} {types}", flush=True)
    rt.contraction(out, rt.upload(a), rt.upload(b), in_t, out_t, *maps)
    assert np.array_equal(out.read(out_t).ravel(), want.ravel())


# Aligned K in rows an odd stride apart, a reordered output, batches, and neighbours of each row's end that
# would make every cell NaN or wrong if they were read as part of it.
LAYOUTS = [("M, K # 101", "N, K", "M, N"), ("M, K", "N, K # 99", "N, M"), ("B, M, K # 97", "B, N, K", "B, M, N"),
           ("M, B, K", "B, N, K", "M, B, N")]


@pytest.mark.parametrize("layout", LAYOUTS, ids=lambda c: " | ".join(c))
@pytest.mark.parametrize("k", [96, 91])
@pytest.mark.parametrize("types", ["bf16-f32", "i8-i32"])
def test_gemm_any_alignment_layouts(rt, layout, k, types):
    l_t, r_t, o_t = layout
    in_t, out_t = TYPES[types]
    s = dict(B=3, M=41, N=70, K=k)
    rng = np.random.default_rng(k)
    axes = dict(B=s["B"] if "B" in l_t else 1)
    av = rng.integers(-2, 3, (axes["B"], s["M"], k))
    bv = rng.integers(-2, 3, (axes["B"], s["N"], k))

    def store(text, v, rows):
        width = int(text.split("# ")[1]) if "#" in text else k
        order = text.split("#")[0].split(", ")
        full = np.full((axes["B"], rows, width), 127.0 if in_t == fh.I8 else np.nan)
        full[:, :, :k] = v
        if order[0] != "B" and "B" in order:
            full = full.transpose(1, 0, 2)
        f = np.ascontiguousarray(full).ravel()
        return f.astype(np.int8) if in_t == fh.I8 else emu.f32_to_bf16(f.astype(np.float32))

    acc = np.einsum("bmk,bnk->bmn", av, bv)
    if o_t == "N, M":
        acc = acc.transpose(0, 2, 1)
    elif o_t == "M, B, N":
        acc = acc.transpose(1, 0, 2)
    pre = ("B, " if "B" in l_t else "") + "M, N, K"
    out = rt.alloc(acc.size * 4)
    print(f"gemm any {layout} K {k} {types}", flush=True)
    rt.contraction(out, rt.upload(store(l_t, av, s["M"])), rt.upload(store(r_t, bv, s["N"])), in_t, out_t,
                   *(fh.m(t, **s) for t in (l_t, r_t, pre, o_t)))
    assert np.array_equal(out.read(out_t).ravel(), narrowed(np.ascontiguousarray(acc).ravel(), out_t).ravel())


# More products or columns than 512 tiles of 64x64, a side of at most 64: the smaller tile.
@pytest.mark.parametrize("size", [(520, 32, 31, 65), (70, 64, 520, 71), (1, 16, 33001, 129)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("types", ["bf16-f32", "i8-i32"])
def test_gemm_any_many_small_exact(rt, size, types):
    b, m, n, k = size
    in_t, out_t = TYPES[types]
    rng = np.random.default_rng(sum(size))
    av, a = operands(rng, in_t, b * m, k)
    bv, w = operands(rng, in_t, b * n, k)
    want = narrowed(np.matmul(av.reshape(b, m, k).astype(np.float64), bv.reshape(b, n, k).astype(np.float64).transpose(0, 2, 1)), out_t)
    maps = [fh.m(t, B=b, M=m, N=n, K=k) for t in ("B, M, K", "B, N, K", "B, M, N, K", "B, M, N")]
    out = rt.upload(np.full(b * m * n, 0x5A, dtype=fh.NP_DTYPE[out_t]))
    print(f"gemm any many {size} {types}", flush=True)
    rt.contraction(out, rt.upload(a), rt.upload(w), in_t, out_t, *maps)
    assert np.array_equal(out.read(out_t).ravel(), want.ravel())
