"""The folds built for one residue wheel (k_contract_wheel, k_reduce_strided and k_reduce_wave by op): around
their read batches, with padded output cells, against the oracle's serial fold, bit for bit where the
order is the serial one."""
import numpy as np
import pytest

import furiosa_hip as fh
from oracle import emulator as emu
from oracle import mapping_ref as mr
from test_gpu_storage import special_bf16

pytestmark = pytest.mark.gpu

F32, BF16 = fh.F32, fh.BF16


@pytest.mark.parametrize("k", [1, 2, 15, 16, 17, 31])
@pytest.mark.parametrize("out", ["N, G, D", "D, N # 5, G", "G # 3, N, D # 24"])
@pytest.mark.parametrize("types", [(BF16, F32), (BF16, BF16), (F32, F32), (fh.I8, fh.I32)], ids=["bf16-f32", "bf16", "f32", "i8"])
def test_contract_one_wheel_exact(rt, types, out, k):
    """A weighted sum's layout: weights [N, G, T], values [T, N, D], K = T strided in the values."""
    in_t, out_t = types
    s = dict(N=3, G=2, D=19, T=k)
    maps = ("N, G, T", "T, N, D", "N, G, D, T", out)
    lo, ro, po, oo = (mr.parse(t, s) for t in maps)
    rng = np.random.default_rng(k)
    if in_t == BF16:
        lhs, rhs = special_bf16(rng, mr.size(lo)), special_bf16(rng, mr.size(ro))
    elif in_t == F32:
        lhs, rhs = (rng.standard_normal(mr.size(o)).astype(np.float32) for o in (lo, ro))
    else:
        lhs, rhs = (rng.integers(-128, 128, mr.size(o)).astype(np.int8) for o in (lo, ro))
    want = emu.contraction(lhs, rhs, in_t, out_t, lo, ro, po, oo)
    dst = rt.upload(np.full(mr.size(oo), 0x5A, dtype=fh.NP_DTYPE[out_t]))  # dead cells must come out zero
    print(f"one-wheel contraction K {k} -> {out} {types}", flush=True)
    rt.contraction(dst, rt.upload(lhs), rt.upload(rhs), in_t, out_t, *(fh.m(t, **s) for t in maps))
    assert np.array_equal(dst.read(out_t).view(np.uint8), want.view(np.uint8))


@pytest.mark.parametrize("r", [1, 31, 32, 33, 63])
@pytest.mark.parametrize("op", ["ADD", "MAX", "MUL"])
@pytest.mark.parametrize("out", ["A, D", "D # 12, A"])
@pytest.mark.parametrize("via_bf16", [False, True], ids=["f32", "rounded"])
def test_reduce_strided_exact(rt, via_bf16, out, op, r):
    s = dict(A=5, R=r, D=11)
    so, do = mr.parse("A, R, D", s), mr.parse(out, s)
    rng = np.random.default_rng(r)
    x = (rng.standard_normal(mr.size(so)) + 0.5).astype(np.float32)
    src = rt.upload(x)
    if via_bf16:  # a widen of a narrow, both deferred: the reduce rounds each element as it reads it
        half, wide = rt.alloc(2 * len(x)), rt.alloc(4 * len(x))
        rt.map(half, BF16, src, F32, len(x), fh.op("CAST"))
        rt.map(wide, F32, half, BF16, len(x), fh.op("CAST"))
        x, src = emu.bf16_to_f32(emu.f32_to_bf16(x)), wide
    ident = {"ADD": 0.0, "MAX": -np.inf, "MUL": 1.0}[op]
    want = emu.reduce(x, F32, so, do, fh.RED[op], fh.f32_bits(ident))
    dst = rt.alloc(4 * mr.size(do))
    print(f"strided reduce {r} {op} -> {out}", flush=True)
    rt.reduce(dst, src, F32, fh.m("A, R, D", **s), fh.m(out, **s), fh.RED[op], fh.f32_bits(ident))
    assert np.array_equal(dst.read(F32).view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("r", [64, 65, 511, 512, 1024, 1100])
@pytest.mark.parametrize("op", ["ADD", "MAX", "MIN"])
def test_reduce_rows_by_op(rt, op, r):
    """Contiguous rows: maxima and minima exact; sums within the n + 4 ulps that any order of n f32
    additions of positive values stays in."""
    s = dict(A=9, R=r)
    rng = np.random.default_rng(r)
    x = rng.uniform(0.5, 1.5, 9 * r).astype(np.float32)
    ident = {"ADD": 0.0, "MAX": -np.inf, "MIN": np.inf}[op]
    dst = rt.alloc(4 * 12)
    rt.reduce(dst, rt.upload(x), F32, fh.m("A, R", **s), fh.m("A # 12", **s), fh.RED[op], fh.f32_bits(ident))
    got = dst.read(F32)
    assert np.array_equal(got[9:], np.full(3, ident, np.float32))
    rows = x.reshape(9, r).astype(np.float64)
    if op == "ADD":
        want = rows.sum(1)
        assert np.all(np.abs(got[:9] - want) <= (r + 4) * np.spacing(want.astype(np.float32)))
    else:
        assert np.array_equal(got[:9], (rows.max(1) if op == "MAX" else rows.min(1)).astype(np.float32))
