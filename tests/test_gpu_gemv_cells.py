"""The GEMV's block sizes (16 cells up to 4096 rows, 32 or 64 past them) around their last blocks, stages of 96
elements and the load ring's rounds, with a strided output: bit for bit against the oracle's serial fold."""
import numpy as np
import pytest

import furiosa_hip as fh
from oracle import emulator as emu
from oracle import mapping_ref as mr
from test_gpu_storage import special_bf16

pytestmark = pytest.mark.gpu

F32, BF16 = fh.F32, fh.BF16


@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 4095, 4096, 4097, 4128, 4129, 8193, 8255, 8256, 8257, 16385])
@pytest.mark.parametrize("k", [8, 96, 104, 392])
@pytest.mark.parametrize("out_t", [F32, BF16])
def test_gemv_cells_exact(rt, n, k, out_t):
    s = dict(N=n, K=k)
    maps = ("K", f"N, K # {k + 8}", "N, K", "N")
    lo, ro, po, oo = (mr.parse(t, s) for t in maps)
    rng = np.random.default_rng(n * 7 + k)
    lhs, rhs = special_bf16(rng, mr.size(lo)), special_bf16(rng, mr.size(ro))
    want = emu.contraction(lhs, rhs, BF16, out_t, lo, ro, po, oo)
    dst = rt.upload(np.full(mr.size(oo), 0x5A, dtype=fh.NP_DTYPE[out_t]))
    print(f"gemv cells {n} x {k} out {out_t}", flush=True)
    rt.contraction(dst, rt.upload(lhs), rt.upload(rhs), BF16, out_t, *(fh.m(t, **s) for t in maps))
    assert np.array_equal(dst.read(out_t).view(np.uint8), want.view(np.uint8))


def test_gemv_most_stages(rt):
    """K = 4096, all of x in LDS: 42 full stages and a part of one."""
    s = dict(N=40, K=4096)
    lo, ro, po, oo = (mr.parse(t, s) for t in ("K", "N, K", "N, K", "N"))
    rng = np.random.default_rng(3)
    lhs, rhs = special_bf16(rng, mr.size(lo)), special_bf16(rng, mr.size(ro))
    want = emu.contraction(lhs, rhs, BF16, F32, lo, ro, po, oo)
    dst = rt.alloc(40 * 4)
    print("gemv K 4096", flush=True)
    rt.contraction(dst, rt.upload(lhs), rt.upload(rhs), BF16, F32, *(fh.m(t, **s) for t in ("K", "N, K", "N, K", "N")))
    assert np.array_equal(dst.read(F32).view(np.uint8), want.view(np.uint8))
