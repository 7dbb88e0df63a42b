"""RMSNorm -> softmax over any row length (k_rmsnorm_softmax_row): each choice of waves per row at the
first, last and ragged columns of its range, rows that start at odd addresses, and the streamed form."""
import numpy as np
import pytest

import furiosa_hip as fh  # noqa: F401  (the library under test)
from oracle import emulator as emu
from test_gpu_fused import bf16, close_chain, rmsnorm_bound, rmsnorm_softmax_numpy

pytestmark = pytest.mark.gpu

SHAPES = [(3, 1), (5, 7), (9, 8), (6, 63), (5, 511), (5, 513), (7, 1001), (3, 1024), (5, 1025), (3, 2047), (2, 2049),
          (3, 4095), (2, 4097), (3, 8191), (2, 8193), (2, 16383), (1, 16385), (2, 32767), (1, 32768), (1, 32769),
          # past 10 MiB a tensor: streamed accesses, two waves a row up to 3072 columns
          (5200, 1025), (3000, 2047), (2601, 2049), (1710, 3072), (1706, 3073), (6144, 4096),
          # the DMA form at 2048 columns, whole and partial last rounds, and one round of 4096
          (7497, 2048), (8192, 2048), (4096, 4096), (3841, 4096)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_rmsnorm_softmax_rows(rt, shape):
    rows, cols = shape
    rng = np.random.default_rng(rows + cols)
    x, g = bf16(rng, rows * cols), bf16(rng, cols, 0.1, 1.0)
    want = rmsnorm_softmax_numpy(x, g, rows, cols, 1e-6)
    out = rt.upload(np.full(rows * cols + 8, 0x5A5A, np.uint16))
    print(f"rmsnorm_softmax rows {rows}x{cols}", flush=True)
    rt.rmsnorm_softmax(out, rt.upload(x), rt.upload(g), rows, cols, 1e-6)
    got = out.read(np.uint16)
    assert np.all(got[rows * cols:] == 0x5A5A)  # nothing past the last row
    close_chain(emu.bf16_to_f32(got[:rows * cols]).reshape(rows, cols), want, hard=rmsnorm_bound(x, g, rows, cols, 1e-6),
                frac_beyond=1e-4)


@pytest.mark.parametrize("cols", [65, 1000, 3001, 5000])
def test_rmsnorm_softmax_rows_nonfinite(rt, cols):
    """A NaN, an infinity and a square past f32's range each send their own row, and no other, through
    the reference's per-element rules; so does a gain of 2^121 every row."""
    rows = 9
    rng = np.random.default_rng(cols)
    x = bf16(rng, rows * cols).reshape(rows, cols)
    x[1, 0], x[3, cols - 1], x[6, 33] = emu.f32_to_bf16(np.array([np.nan, np.inf, 1e20], np.float32))
    for huge in (False, True):
        g = bf16(rng, cols, 0.1, 1.0)
        if huge:
            g[cols - 2] = emu.f32_to_bf16(np.array([2.0 ** 121], np.float32))[0]
        want = emu.bf16_to_f32(emu.rmsnorm_softmax(x.ravel(), g, rows, cols, 1e-6)).reshape(rows, cols)
        out = rt.alloc(rows * cols * 2)
        rt.rmsnorm_softmax(out, rt.upload(x.ravel()), rt.upload(g), rows, cols, 1e-6)
        got = emu.bf16_to_f32(out.read(np.uint16)).reshape(rows, cols)
        assert np.array_equal(np.isnan(got), np.isnan(want))
        fin = ~np.isnan(want)
        assert fin[[0, 2, 4, 5, 7, 8]].all() and np.isnan(want[[1, 3]]).all()
        if not huge:
            bound = rmsnorm_bound(x.ravel(), g, rows, cols, 1e-6)
            close_chain(got[fin], want[fin], frac_beyond=1e-4, hard=bound[fin])


@pytest.mark.parametrize("shape", [(3, 512), (3, 999), (6144, 4096), (3, 32000), (3, 32768)], ids=lambda s: "x".join(map(str, s)))
def test_rmsnorm_softmax_rows_large_gain(rt, shape):
    """One nonzero value a row against gains up to where y overflows: y is the largest a finite row gives,
    sqrt(cols) times the gain, and its softmax is one there and zero elsewhere."""
    rows, cols = shape
    x = np.zeros((rows, cols), np.float32)
    x[:, 17] = 1.0
    x[1, 17], x[1, cols - 1], x[2, 17] = 0.0, 3.0, -1.0
    x = emu.f32_to_bf16(x.ravel())
    for gain in (2.0 ** 20, 2.0 ** 21, 2.0 ** 24 * 1.5, 2.0 ** 60, 2.0 ** 119 * 1.9921875, 2.0 ** 120):
        g = emu.f32_to_bf16(np.full(cols, gain, np.float32))
        want = emu.bf16_to_f32(emu.rmsnorm_softmax(x[:3 * cols], g, 3, cols, 1e-6)).reshape(3, cols)
        assert want[0, 17] == 1.0 and want[1, cols - 1] == 1.0 and want[2, 17] == 0.0
        out = rt.alloc(rows * cols * 2)
        print(f"rmsnorm_softmax large gain {shape} {gain}", flush=True)
        rt.rmsnorm_softmax(out, rt.upload(x), rt.upload(g), rows, cols, 1e-6)
        got = emu.bf16_to_f32(out.read(np.uint16)).reshape(rows, cols)
        assert np.array_equal(got[:2], want[:2]) and np.all(got[3:] == want[0])
        # the third row's equal weights are 1 / (cols - 1) each, within a rounding to bf16 either way
        assert np.all(np.abs(got[2] - want[2]) <= 2.0 ** -7 * want[2])


@pytest.mark.parametrize("shape", [(3, 64), (3, 500), (3, 1024), (3, 5000), (2, 20000), (6144, 4096)], ids=lambda s: "x".join(map(str, s)))
def test_rmsnorm_softmax_rows_no_mean_square(rt, shape):
    """Without an eps, a row of zeros and a row whose squares all flush to zero divide by zero: their outputs
    are the reference's NaN, bit for bit."""
    rows, cols = shape
    x = np.full((rows, cols), 0x3F80, np.uint16)
    x[0], x[rows - 1] = 0, 0x8080  # zeros; the smallest normal bf16, negative
    x[rows - 1, 0] = 0x0080
    g = emu.f32_to_bf16(np.ones(cols, np.float32))
    want = emu.rmsnorm_softmax(x[[0, 1, rows - 1]].ravel(), g, 3, cols, 0.0).reshape(3, cols)
    out = rt.alloc(rows * cols * 2)
    print(f"rmsnorm_softmax no mean square {rows}x{cols}", flush=True)
    rt.rmsnorm_softmax(out, rt.upload(x.ravel()), rt.upload(g), rows, cols, 0.0)
    got = out.read(np.uint16).reshape(rows, cols)
    assert np.all(want[[0, 2]] == 0x7FC0) and np.array_equal(got[[0, rows - 1]], want[[0, 2]])
    if rows > 2:
        assert np.array_equal(got[1], want[1])


def test_rmsnorm_softmax_rows_past_one_launch(rt):
    """More rows than one launch's threads reach (2^25 at 64 threads a row): the second launch continues where
    the first ended."""
    rows, cols, part = 2 ** 25 + 5, 2, 4096
    rng = np.random.default_rng(25)
    x, g = bf16(rng, 3 * part * cols), bf16(rng, cols, 0.1, 1.0)
    whole = np.resize(x, rows * cols)
    out = rt.alloc(rows * cols * 2)
    print(f"rmsnorm_softmax past one launch {rows}x{cols}", flush=True)
    rt.rmsnorm_softmax(out, rt.upload(whole), rt.upload(g), rows, cols, 1e-6)
    got = out.read(np.uint16).reshape(rows, cols)
    want = rmsnorm_softmax_numpy(x, g, 3 * part, cols, 1e-6)
    close_chain(emu.bf16_to_f32(got[:3 * part].ravel()).reshape(-1, cols), want, hard=rmsnorm_bound(x, g, 3 * part, cols, 1e-6),
                frac_beyond=1e-4)
    assert np.array_equal(got, np.resize(got[:3 * part], got.shape))
