"""The tile sizes of the MFMA contraction (k_gemm, k_gemm4) and the blocks that share an output tile.

Operands are small integers, exact in every operand type, and every product and partial sum is a
small integer too, so any order of summation gives the same result: outputs are compared bit for bit
with the integer product."""
import numpy as np
import pytest

import furiosa_hip as fh
from oracle import emulator as emu

pytestmark = pytest.mark.gpu

TYPES = {"bf16": (fh.BF16, fh.BF16), "bf16-f32": (fh.BF16, fh.F32), "i8": (fh.I8, fh.I8), "i8-i32": (fh.I8, fh.I32),
         "e4m3-f32": (fh.F8E4M3, fh.F32), "e5m2": (fh.F8E5M2, fh.F8E5M2)}


def operands(rng, in_t, rows, k):
    v = rng.integers(-2, 3, (rows, k))
    if in_t == fh.I8:
        return v, v.astype(np.int8)
    f = v.astype(np.float32).ravel()
    return v, emu.f32_to_bf16(f) if in_t == fh.BF16 else emu.f32_to_f8(f, in_t)


def narrowed(acc, out_t):
    """The integer sums as the output type's elements, by the output type's own narrow."""
    if out_t in (fh.I8, fh.I32):
        return acc.astype(np.int64).astype(fh.NP_DTYPE[out_t])  # wraps
    f = acc.astype(np.float32).ravel()
    return f if out_t == fh.F32 else emu.f32_to_bf16(f) if out_t == fh.BF16 else emu.f32_to_f8(f, out_t)


def product(a, b):
    return a.astype(np.float64) @ b.astype(np.float64).T  # exact: |sum| < 2^53


# One tile and its remainders, K below, at and past a stage; then sizes where 8, 4, 3 and 2 blocks
# share a tile (uneven runs of stages, a partial last one); then the first and last sizes of each tile, four
# stages in flight among them, and small sides past 512 tiles.
SIZES = [(8, 8, 16), (64, 64, 64), (65, 63, 80), (9, 70, 6160), (64, 64, 12304), (130, 200, 4624), (128, 1030, 2080),
         (257, 8136, 512), (520, 4096, 144), (2048, 2049, 96), (2300, 4090, 64), (3072, 3000, 48),
         (257, 8136, 1552), (257, 8136, 2320), (20, 33000, 80), (33010, 63, 48), (33000, 40, 272), (70, 70000, 48)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("types", list(TYPES))
def test_gemm_tiles_exact(rt, size, types):
    m, n, k = size
    in_t, out_t = TYPES[types]
    rng = np.random.default_rng(m + n + k)
    av, a = operands(rng, in_t, m, k)
    bv, b = operands(rng, in_t, n, k)
    want = narrowed(product(av, bv), out_t)
    maps = [fh.m(t, M=m, N=n, K=k) for t in ("M, K", "N, K", "M, N, K", "M, N")]
    out = rt.upload(np.full(m * n, 0x5A, dtype=fh.NP_DTYPE[out_t]))
    da, db = rt.upload(a), rt.upload(b)
    print(f"gemm tiles {size} {types}", flush=True)
    for _ in range(2):  # the second launch finds the arrival counters the first left
        rt.contraction(out, da, db, in_t, out_t, *maps)
        assert np.array_equal(out.read(out_t).ravel(), want.ravel())


def test_gemm_shared_tiles_batched_and_transposed(rt):
    """Batch cells and a transposed output with several blocks a tile."""
    B, m, n, k = 3, 40, 72, 3200
    rng = np.random.default_rng(5)
    av, a = operands(rng, fh.BF16, B * m, k)
    bv, b = operands(rng, fh.BF16, B * n, k)
    want = np.stack([product(x, y).T for x, y in zip(av.reshape(B, m, k), bv.reshape(B, n, k))])
    maps = [fh.m(t, B=B, M=m, N=n, K=k) for t in ("B, M, K", "B, N, K", "B, M, N, K", "B, N, M")]
    out = rt.alloc(B * m * n * 4)
    rt.contraction(out, rt.upload(a), rt.upload(b), fh.BF16, fh.F32, *maps)
    assert np.array_equal(out.read(fh.F32), narrowed(want, fh.F32))


@pytest.mark.parametrize("size", [(1, 256, 4096), (16, 1000, 8192), (33, 640, 1040)], ids=lambda s: "x".join(map(str, s)))
def test_w8a8_shared_tiles(rt, size):
    """The dequant epilogue and the raw accumulators with several blocks a tile, eagerly and over
    replays of a recorded graph with other work between."""
    m, n, k = size
    rng = np.random.default_rng(k)
    av, bv = rng.integers(-127, 128, (m, k)), rng.integers(-127, 128, (n, k))
    scale = rng.uniform(1e-3, 1e-2, n).astype(np.float32)
    acc = product(av, bv)
    want = emu.f32_to_bf16((acc.astype(np.float32) * scale).ravel())
    a, w, s = rt.upload(av.astype(np.int8)), rt.upload(bv.astype(np.int8)), rt.upload(scale)
    out, raw = rt.alloc(m * n * 2), rt.alloc(m * n * 4)
    rt.gemm_w8a8_dequant(out, raw, a, w, s, m, n, k)
    assert np.array_equal(out.read(np.uint16), want)
    assert np.array_equal(raw.read(np.int32), acc.astype(np.int32).ravel())
    other = rt.alloc(m * n * 2)
    rt.graph_begin()
    rt.gemm_w8a8_dequant(out, None, a, w, s, m, n, k)
    graph = rt.graph_end()
    for _ in range(4):
        out.write(np.zeros(m * n, np.uint16))
        graph.launch()
        assert np.array_equal(out.read(np.uint16), want)
        rt.gemm_w8a8_dequant(other, None, a, w, s, m, n, k)
        assert np.array_equal(other.read(np.uint16), want)
    graph.free()


# Batches of products smaller than a tile, more of them than 512 tiles.
@pytest.mark.parametrize("size", [(520, 16, 64, 80), (600, 63, 40, 48), (530, 100, 72, 160)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("types", list(TYPES))
def test_gemm_tiles_batches_exact(rt, size, types):
    b, m, n, k = size
    in_t, out_t = TYPES[types]
    rng = np.random.default_rng(sum(size))
    av, a = operands(rng, in_t, b * m, k)
    bv, w = operands(rng, in_t, b * n, k)
    want = narrowed(np.matmul(av.reshape(b, m, k).astype(np.float64), bv.reshape(b, n, k).astype(np.float64).transpose(0, 2, 1)), out_t)
    maps = [fh.m(t, B=b, M=m, N=n, K=k) for t in ("B, M, K", "B, N, K", "B, M, N, K", "B, M, N")]
    out = rt.upload(np.full(b * m * n, 0x5A, dtype=fh.NP_DTYPE[out_t]))
    print(f"gemm tiles batches {size} {types}", flush=True)
    rt.contraction(out, rt.upload(a), rt.upload(w), in_t, out_t, *maps)
    assert np.array_equal(out.read(out_t).ravel(), want.ravel())
