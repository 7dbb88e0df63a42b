"""Attention with a step's keys split over wave groups (k_attn_split): both forms and the 256-query form on
either side of their rule, at the edges of query groups, key blocks and steps."""
import numpy as np
import pytest

from oracle import emulator as emu
from test_gpu_fused import attention_numpy, bf16, close_chain

pytestmark = pytest.mark.gpu

# (heads, seq): the 4 x 2 form up to 64 keys, the 2 x 4 form over several steps of 256 keys, then the 4 x 2 form (more
# than 256 workgroups of 64 queries, at most 256 to 512 of 128 by length and mask), then the 256-query form: one
# query block, several with a ragged last one.
CASES = [(1, 1), (3, 31), (2, 32), (5, 33), (2, 63), (2, 64), (3, 65), (2, 129), (1, 255), (2, 256), (1, 257), (2, 511),
         (1, 513), (1, 800), (257, 40), (100, 150), (64, 257), (52, 513), (36, 1025), (330, 90), (170, 333), (110, 600)]


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_attention_split(rt, case, d, causal):
    h, s = case
    sqrt_d = np.float32(8.0 if d == 64 else 11.313708)
    rng = np.random.default_rng(h * 10007 + s)
    q, k, v = (bf16(rng, h * s * d) for _ in range(3))
    out = rt.upload(np.full(h * s * d + 8, 0x5A5A, np.uint16))
    print(f"attention split {h}x{s}x{d} causal={causal}", flush=True)
    rt.attention_prefill(out, rt.upload(q), rt.upload(k), rt.upload(v), 1, h, s, d, float(sqrt_d), causal)
    raw = out.read(np.uint16)
    assert np.all(raw[h * s * d:] == 0x5A5A)  # nothing past the last query
    got = emu.bf16_to_f32(raw[:h * s * d]).reshape(h, s, d)
    heads = range(h) if h <= 5 else sorted(set(int(x) for x in np.linspace(0, h - 1, 5)))
    for i in heads:
        sl = slice(i * s * d, (i + 1) * s * d)
        ref, bound = attention_numpy(q[sl], k[sl], v[sl], s, d, sqrt_d, causal)
        close_chain(got[i], ref, frac_beyond=2e-3, hard=bound)


@pytest.mark.parametrize("h", [2, 110])  # the 2 x 4 form, and several blocks of the 256-query form
def test_attention_split_growing_logits(rt, h):
    """Keys whose logits grow along the sequence, so every later block raises the running max by far
    more than the rescale margin, and queries that see only the first, small ones."""
    s, d = 600, 128
    rng = np.random.default_rng(9)
    q = np.abs(rng.standard_normal((h, s, d))).astype(np.float32)
    k = (rng.standard_normal((h, s, d)) * 0.1 + np.linspace(0.0, 3.0, s)[None, :, None]).astype(np.float32)
    q, k = emu.f32_to_bf16(q.ravel()), emu.f32_to_bf16(k.ravel())
    v = bf16(rng, h * s * d)
    out = rt.alloc(h * s * d * 2)
    rt.attention_prefill(out, rt.upload(q), rt.upload(k), rt.upload(v), 1, h, s, d, 11.313708, True)
    got = emu.bf16_to_f32(out.read(np.uint16)).reshape(h, s, d)
    # a causal row's own max: the chain over its visible keys alone (p rounds at that scale here)
    for i in (0, h - 1):
        sl = slice(i * s * d, (i + 1) * s * d)
        for row in (0, 40, 64, 255, 256, 400, 599):
            n = row + 1
            qs, ks, vs = (t[sl].reshape(s, d)[:n].ravel() for t in (q, k, v))
            ref, bound = attention_numpy(qs, ks, vs, n, d, np.float32(11.313708), False)
            close_chain(got[i, row], ref[row], frac_beyond=2e-2, hard=bound[row])


# One shape of each form, with more than one key block where the form has several: 4 x 2 groups, 2 x 4,
# 4 x 2 over three query blocks, 256 queries.
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("case", [(2, 64), (2, 600), (64, 300), (170, 333)], ids=lambda c: "x".join(map(str, c)))
def test_attention_infinite_logits(rt, case, d, causal):
    """Without a row max given, every form has the same result for logits that overflow: a -inf logit's key
    weighs nothing (a whole first block of them too), and a row is NaN where it sees a +inf or a NaN logit
    or no logit but -inf. Head 0's first keys give -inf to some queries; in head 1 every key does."""
    h, s = case
    sd = np.float32(8.0 if d == 64 else 11.313708)
    rng = np.random.default_rng(h + s + d)
    q, k, v = (bf16(rng, h * s * d).reshape(h, s, d) for _ in range(3))
    big, nan = emu.f32_to_bf16(np.array([2.0 ** 100, np.nan], np.float32))
    minus = big | 0x8000
    first = 20 if s == 64 else 70  # more than one 64-key block
    q[:2, :, 0] = k[:2, :, 0] = 0
    k[0, :first, 0], k[1, :, 0] = big, big
    q[0, [5, 40, s - 1], 0] = q[1, 7, 0] = minus
    q[0, 9, 0], q[0, 11, 1] = big, nan
    out = rt.upload(np.full(h * s * d, 0x5A5A, np.uint16))
    print(f"attention infinite logits {case} d {d} causal={causal}", flush=True)
    rt.attention_prefill(out, *(rt.upload(t.ravel()) for t in (q, k, v)), 1, h, s, d, float(sd), causal)
    got = emu.bf16_to_f32(out.read(np.uint16)).reshape(h, s, d)
    for i in range(2):
        with np.errstate(all="ignore"):  # inf and NaN logits
            qf, kf, vf = (emu.bf16_to_f32(t[i].ravel()).reshape(s, d).astype(np.float64) for t in (q, k, v))
            x = qf @ kf.T / sd
            x[np.abs(x) > 3e38] *= np.inf
            if causal:
                x[~np.tri(s, dtype=bool)] = -np.inf
            e = np.exp(x - x.max(axis=1, keepdims=True))
            ref = e @ vf / e.sum(axis=1, keepdims=True)
        bad = {9, 11} | ({5, 40} if causal and s > 64 else {5} if causal else set()) if i == 0 else {7}
        assert set(np.flatnonzero(np.isnan(ref).any(axis=1))) == bad
        assert np.array_equal(np.isnan(got[i]), np.isnan(ref))
        ok = [r for r in range(s) if r not in bad]
        # logits below 8 round to bf16 within 2^-6, so each weight moves by at most e^(2^-6) either way and an
        # average by 2^-5 of the values' size; the roundings of p, of o and of the result are 2^-7 of it
        assert np.all(np.abs(got[i][ok] - ref[ok]) <= (2.0 ** -5 + 2.0 ** -7) * np.abs(vf).max())
