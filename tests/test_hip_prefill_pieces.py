"""Attention of many query rows on the matrix cores, operands in pieces of bfloat16: heads that are no whole row tiles, caches
that end within a tile of keys, keys cut over workgroups, values that must go to the 32-bit instructions."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("far", ["", "tiny V", "huge V", "huge K"])
@pytest.mark.parametrize("S,pos0", [(33, 0), (128, 0), (160, 31), (257, 70), (512, 3)])
@pytest.mark.parametrize("hd,rep", [(64, 4), (64, 3), (128, 2), (128, 5)])
def test_against_64_bits(hip, hd, rep, S, pos0, far):
    rng = np.random.default_rng(hd + rep + S)
    B, kvh, T = 2, 2, pos0 + S
    q, k, v = (rng.standard_normal(s, dtype=np.float32) for s in ((B, kvh * rep, S, hd), (B, kvh, T, hd), (B, kvh, T, hd)))
    if far == "tiny V":
        v[..., 4:9] *= np.float32(1e-31)
    elif far == "huge V":
        v[:, :, T // 2, 7] = np.float32(3.2e38)
    elif far == "huge K":
        k, q = k * np.float32(2.0 ** 66), q * np.float32(2.0 ** -66)
    got = hip.to_numpy(cases.decode_attention_ops(hip, hip.from_numpy(q), hip.from_numpy(k), hip.from_numpy(v), rep))
    q, k, v = (x.astype(np.float64) for x in (q, np.repeat(k, rep, 1), np.repeat(v, rep, 1)))
    s = np.matmul(q, k.transpose(0, 1, 3, 2)) / np.sqrt(hd)
    s[..., np.arange(T)[None, :] > pos0 + np.arange(S)[:, None]] = -np.inf
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    # scores: a rounding per product and sum; a weight is off by twice that (its own and the largest score's), by the rounding of
    # the exponent's argument (below 32) and the exponential's; then a rounding per key in the sum and in the weighted sum
    score = (hd + 8) * 2.0 ** -24 * (np.matmul(np.abs(q), np.abs(k).transpose(0, 1, 3, 2)) / np.sqrt(hd)).max(-1, keepdims=True)
    bound = (2 * score + 64 * 2.0 ** -24 + 2 * (T + 16) * 2.0 ** -24) * np.matmul(p, np.abs(v))
    err = np.abs(got - np.matmul(p, v))
    print("error / bound: max %.3f, mean %.5f" % ((err / bound).max(), (err / bound).mean()), flush=True)
    assert (err <= bound).all()


@pytest.mark.parametrize("hd,rep,S", [(64, 3, 512), (64, 4, 1500), (128, 2, 1024)])
def test_roundings_have_no_direction(hip, hd, rep, S):
    """The outputs' error in the mean, against their root mean square per query: roundings to nearest have none (over these numbers of
    outputs below 2^-28), sums that are cut off below have 2^-26 and more."""
    rng = np.random.default_rng(S)
    q, k, v = (rng.standard_normal(s, dtype=np.float32) for s in ((2, 4 * rep, S, hd), (2, 4, S, hd), (2, 4, S, hd)))
    got = hip.to_numpy(cases.decode_attention_ops(hip, hip.from_numpy(q), hip.from_numpy(k), hip.from_numpy(v), rep))
    q, k, v = (x.astype(np.float64) for x in (q, np.repeat(k, rep, 1), np.repeat(v, rep, 1)))
    s = np.matmul(q, k.transpose(0, 1, 3, 2)) / np.sqrt(hd)
    s[..., np.triu(np.ones((S, S), dtype=bool), 1)] = -np.inf
    p = np.exp(s - s.max(-1, keepdims=True))
    want = np.matmul(p / p.sum(-1, keepdims=True), v)
    d = (got - want) / np.sqrt((want ** 2).mean(-1, keepdims=True))
    assert abs(d.mean()) <= 2.0 ** -28, d.mean()


@pytest.mark.parametrize("hd,rep,S", [(64, 3, 200), (128, 2, 140)])
@pytest.mark.parametrize("low,high", [(-149, -126), (-126, -115), (-149, 3), (80, 95)])
def test_values_of_any_size(hip, hd, rep, S, low, high):
    """V with small (or very large) values beside ordinary ones: queries that see only such keys get all of their bits."""
    rng = np.random.default_rng(S + high)
    q, k, v = (rng.standard_normal(s, dtype=np.float32) for s in ((1, 2 * rep, S, hd), (1, 2, S, hd), (1, 2, S, hd)))
    v[:, :, :70, ::3] = np.ldexp(v[:, :, :70, ::3], rng.integers(low, high, v[:, :, :70, ::3].shape)).astype(np.float32)
    got = hip.to_numpy(cases.decode_attention_ops(hip, hip.from_numpy(q), hip.from_numpy(k), hip.from_numpy(v), rep))
    q, k, v = (x.astype(np.float64) for x in (q, np.repeat(k, rep, 1), np.repeat(v, rep, 1)))
    s = np.matmul(q, k.transpose(0, 1, 3, 2)) / np.sqrt(hd)
    s[..., np.triu(np.ones((S, S), dtype=bool), 1)] = -np.inf
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    score = (hd + 8) * 2.0 ** -24 * (np.matmul(np.abs(q), np.abs(k).transpose(0, 1, 3, 2)) / np.sqrt(hd)).max(-1, keepdims=True)
    # as above, and the spacing of subnormal numbers per key and step of the division
    bound = (2 * score + 64 * 2.0 ** -24 + 2 * (S + 16) * 2.0 ** -24) * np.matmul(p, np.abs(v)) + (S + 8) * 2.0 ** -149
    assert (np.abs(got - np.matmul(p, v)) <= bound).all()
