"""Relayouts of ragged sizes: tiled transposes whose rows start at any element address (k_relayout_tiled16's
general form) and contiguous runs of any length (k_relayout_runs), against the oracle, byte for byte."""
import numpy as np
import pytest

import furiosa_hip as fh
from oracle import emulator as emu
from oracle import mapping_ref as mr

pytestmark = pytest.mark.gpu

DTYPES = {"i8": (fh.I8, np.int8), "bf16": (fh.BF16, np.uint16), "f32": (fh.F32, np.int32)}

CASES = [
    # transposes: one tile, tile edges, odd rows, batches, a live prefix of either tile axis, a broadcast
    (dict(A=16, B=17), "A, B", "B, A"),
    (dict(A=63, B=65), "A, B", "B, A"),
    (dict(A=129, B=64), "A, B", "B, A"),
    (dict(A=300, B=111), "A, B", "B, A"),
    (dict(A=33, B=5, C=47), "A, B, C", "C, B, A"),
    (dict(A=33, B=5, C=47), "A, B, C", "B, C, A"),
    (dict(A=37, B=70), "A, B # 75", "B, A # 41"),
    (dict(A=37, B=70), "A # 40, B", "B # 72, A"),
    (dict(A=21, B=35, X=3), "A, B", "X, B, A"),
    (dict(A=21, B=35, X=3), "A, B", "B, X, A # 24"),
    # runs: shorter than, equal to and past a piece, odd addresses, padded, broadcast
    (dict(A=9, B=7, C=8), "A, B, C", "B, A, C"),
    (dict(A=9, B=7, C=9), "A, B, C", "B, A, C"),
    (dict(A=9, B=7, C=16), "A, B, C # 17", "B, A, C"),
    (dict(A=5, B=40, C=100), "A, B, C", "B, A, C # 103"),
    (dict(A=5, B=4, C=333), "A # 6, B, C", "B, A, C"),
    (dict(A=11, C=23, X=4), "A, C", "X, A, C # 25"),
    (dict(A=3, B=2, C=1001), "A, B, C", "B, A # 5, C"),
]


@pytest.mark.parametrize("case", CASES, ids=[f"{c[1]} -> {c[2]}: {c[0]}" for c in CASES])
@pytest.mark.parametrize("dt", list(DTYPES))
def test_relayout_ragged(rt, case, dt):
    sizes, s_t, d_t = case
    t, npt = DTYPES[dt]
    rng = np.random.default_rng(len(s_t) + sum(sizes.values()))
    so, do = mr.parse(s_t, sizes), mr.parse(d_t, sizes)
    info = np.iinfo(npt)
    src = rng.integers(info.min, info.max, mr.size(so), dtype=npt, endpoint=True)
    init = rng.integers(info.min, info.max, mr.size(do), dtype=npt, endpoint=True)  # padding keeps its bytes
    want = emu.transpose(init.copy(), src, so, do)
    dst = rt.upload(init)
    print(f"relayout {sizes} {s_t} -> {d_t} {dt}", flush=True)
    rt.transpose(dst, rt.upload(src), t, fh.m(s_t, **sizes), fh.m(d_t, **sizes), allow_broadcast="X" in d_t)
    assert np.array_equal(dst.read(npt), want)
