"""The small one-element-a-lane maps and zips (n up to 32768) against the oracle, bit for bit, at the block
and rule edges: every float op both ways round, on signed zeros, infinities, NaN, f32 subnormals and the
narrow's ties."""
import numpy as np
import pytest

import furiosa_hip as fh
from oracle import emulator as emu

pytestmark = pytest.mark.gpu

F32, BF16 = fh.F32, fh.BF16
SIZES = [1, 63, 64, 65, 32768, 32769]
BINARY = ["ADD_F", "CLIP_ADD", "SUB_F", "MUL_F", "DIV_F", "CLIP_MIN", "CLIP_MAX"]


def values(rng, n):
    v = (rng.standard_normal(n) * 3).astype(np.float32)
    odd = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1e-40, -3e-39, 1.00390625, 3.3e38], np.float32)
    at = rng.random(n) < 0.1
    v[at] = rng.choice(odd, int(at.sum()))
    return v


def same(got, want, zeros=False):
    """Bit for bit (a NaN as any NaN); with `zeros`, either zero for either: the sign of the minimum or
    maximum of +0 and -0 is unspecified (f32::min, fminf), and libm and the GPU differ on it."""
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    got, want = got[~nan], want[~nan]
    if zeros:
        assert np.array_equal(got, want)
    else:
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("swap", [0, fh.SWAP], ids=["", "swapped"])
@pytest.mark.parametrize("name", BINARY)
def test_small_binary(rt, name, swap, n):
    rng = np.random.default_rng(n)
    a, b = values(rng, n), values(rng, n)
    da, db, out = rt.upload(a), rt.upload(b), rt.alloc(4 * n)
    rt.zip_with(out, F32, da, db, F32, n, fh.op(name, swap))
    zeros = name in ("CLIP_MIN", "CLIP_MAX")
    same(out.read(F32), emu.zip_(a, b, F32, F32, fh.OP[name], swap), zeros)
    imm = float(np.float32(-0.3125))
    rt.map(out, F32, da, F32, n, fh.op(name, fh.RHS_IMM | swap, imm))
    same(out.read(F32), emu.map_(a, F32, F32, fh.OP[name], swap, fh.f32_bits(imm)), zeros)


@pytest.mark.parametrize("n", SIZES)
def test_small_unary_and_narrow(rt, n):
    rng = np.random.default_rng(n + 1)
    a = values(rng, n)
    da, out, half = rt.upload(a), rt.alloc(4 * n), rt.alloc(2 * n)
    rt.map(half, BF16, da, F32, n, fh.op("CAST"))
    assert np.array_equal(half.read(np.uint16), emu.map_(a, F32, BF16, fh.OP["CAST"]))
    rt.map(out, F32, da, F32, n, fh.op("SQRT"))
    same(out.read(F32), emu.map_(a, F32, F32, fh.OP["SQRT"]))
    x = np.clip(np.nan_to_num(a), -30, 30).astype(np.float32)
    dx = rt.upload(x)
    for name in ("EXP", "NEG_EXP", "SIGMOID"):  # libm against ROCm's: both faithfully rounded
        rt.map(out, F32, dx, F32, n, fh.op(name))
        want = emu.map_(x, F32, F32, fh.OP[name])
        assert np.all(np.abs(out.read(F32) - want) <= 2 * np.spacing(np.abs(want)) + 1e-30)


@pytest.mark.parametrize("n", [1, 96, 24576])
def test_small_zip_reads_deferred_inputs(rt, n):
    """A swapped zip of a broadcast through three deferred maps (one of them reversed) and the widen of a
    deferred narrow: the same bits as with every intermediate written."""
    rng = np.random.default_rng(n + 2)
    rows, cols = (n, 1) if n == 1 else (n // 96, 96)
    s = dict(R=rows, C=cols)
    a, b = np.abs(values(rng, rows)) + np.float32(0.5), values(rng, n)
    a[~np.isfinite(a)] = 2.0
    got = []
    for flush in (False, True):
        keep = []

        def step(buf):
            keep.append(buf)
            if flush:
                buf.flush()
            return buf

        def mapped(x, src_t, dst_t, m, op):
            out = rt.alloc(m * (2 if dst_t == BF16 else 4))
            rt.map(out, dst_t, x, src_t, m, op)
            return step(out)

        x = rt.upload(a)
        x = mapped(x, F32, F32, rows, fh.op("DIV_F", fh.RHS_IMM | fh.SWAP, 3.0))
        x = mapped(x, F32, F32, rows, fh.op("CLIP_ADD", fh.RHS_IMM, 0.25))
        x = mapped(x, F32, F32, rows, fh.op("SQRT"))
        wide = rt.alloc(4 * n)
        rt.transpose(wide, x, F32, fh.m("R", **s), fh.m("R, C", **s), allow_broadcast=True)
        step(wide)
        y = mapped(mapped(rt.upload(b), F32, BF16, n, fh.op("CAST")), BF16, F32, n, fh.op("CAST"))
        out = rt.alloc(4 * n)
        rt.zip_with(out, F32, wide, y, F32, n, fh.op("SUB_F", fh.SWAP))
        got.append(out.read(F32))
    same(got[0], got[1])
