"""The MLP chain for any widths and batches (k_mlp_rows, and its rule against the one-row forms): logits and
argmax bit for bit against the oracle, on inputs with subnormals, signed zeros and exact ties."""
import numpy as np
import pytest

import furiosa_hip as fh
from oracle import emulator as emu
from test_gpu_storage import special_bf16

pytestmark = pytest.mark.gpu

# batch, inputs, hidden, outputs: each rows-per-block choice with a partial last block, odd widths,
# units at and past the powers of two, more units than a block stages at once, the one-row forms' edges.
SHAPES = [(1, 31, 100, 2), (3, 129, 16, 64), (2, 100, 1024, 63), (5, 33, 513, 17), (256, 72, 130, 9), (257, 72, 130, 9),
          (513, 65, 33, 16), (1025, 40, 64, 10), (2049, 24, 128, 5), (2050, 33, 257, 10), (2100, 1000, 512, 64),
          (300, 1024, 20, 33), (512, 72, 64, 9), (513, 72, 64, 9), (257, 72, 65, 9), (1, 4000, 1024, 64), (7, 100, 28, 3),
          # both sides of the lines between the one-row forms and k_mlp_rows
          (3, 72, 200, 5), (3, 72, 201, 5), (257, 80, 80, 7), (257, 81, 79, 7), (400, 256, 128, 9), (512, 131, 65, 9),
          (1000, 100, 100, 50), (600, 161, 33, 16), (1025, 100, 60, 10), (1500, 73, 90, 10), (2048, 73, 23, 34), (2049, 73, 23, 34),
          (362, 123, 17, 50), (300, 131, 131, 50)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_mlp_rows_exact(rt, shape):
    batch, i, h, o = shape
    rng = np.random.default_rng(batch + i + h + o)

    def weights(n, scale):
        w = special_bf16(rng, n)  # with subnormals, zeros and a few large values
        small = rng.random(n) < 0.97
        w[small] = emu.f32_to_bf16((rng.standard_normal(n) * scale).astype(np.float32))[small]
        return w

    x = weights(batch * i, 1.0)
    w1, b1, w2, b2 = weights(h * i, 0.05), weights(h, 0.05), weights(o * h, 0.05), weights(o, 0.05)
    w2.reshape(o, h)[-1] = w2.reshape(o, h)[0]  # equal logits: the last of them wins
    b2[-1] = b2[0]
    rows = sorted(set(np.linspace(0, batch - 1, min(batch, 40)).astype(int)))
    pred, logits = emu.mlp(x.reshape(batch, i)[rows].ravel(), w1, b1, w2, b2, len(rows), i, h, o)
    dp, dl = rt.upload(np.full(batch + 4, -7, np.int32)), rt.upload(np.full(batch * o + 8, 0x5A5A, np.uint16))
    print(f"mlp rows {shape}", flush=True)
    dev = [rt.upload(a) for a in (x, w1, b1, w2, b2)]
    for with_logits in (True, False):
        rt.mlp(dp, dl if with_logits else None, *dev, batch, i, h, o)
        got = dp.read(np.int32)
        assert np.array_equal(got[:batch][rows], pred) and np.all(got[batch:] == -7)
    got = dl.read(np.uint16)
    assert np.array_equal(got[:batch * o].reshape(batch, o)[rows], logits.reshape(-1, o))
    assert np.all(got[batch * o:] == 0x5A5A)


def test_mlp_refuses_widths_past_the_budget(rt):
    buf = rt.alloc(1 << 20)
    with pytest.raises(fh.FoError, match="LDS budget"):
        rt.mlp(buf, None, buf, buf, buf, buf, buf, 1, 16390, 17, 5)
