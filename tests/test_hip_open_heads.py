"""Decode-time attention that norms and embeds the heads of q and of the cache's newest row itself, on every kernel that can and beside those that
leave it to a launch of its own, against float64: a step that appends by copying the caches and one that appends in place."""
import numpy as np
import pytest

import cases
from backends import backend_with_env

pytestmark = pytest.mark.gpu

K, EPS = 516, 1e-5
# (sequences, KV heads, query heads a KV head, head size, cached positions, always in segments)
STEPS = [
    (1, 8, 2, 128, 1, False), (1, 8, 2, 128, 159, False), (1, 8, 2, 128, 160, False), (3, 2, 2, 128, 319, False), (1, 8, 2, 128, 470, False),
    (1, 1, 8, 128, 600, False), (1, 3, 3, 64, 320, False), (2, 3, 1, 64, 640, False), (1, 3, 3, 64, 960, False), (1, 1, 8, 64, 1100, False),  # a row a workgroup
    (3, 3, 1, 64, 4099, False),  # ... in two segments
    (1, 8, 2, 128, 1030, False), (4, 8, 2, 128, 700, False), (1, 3, 3, 64, 1024, True), (1, 1, 6, 64, 1023, True), (2, 1, 8, 128, 1025, True),  # segments
    (8, 8, 2, 128, 700, True), (8, 8, 5, 64, 1030, True),  # ... of several trips
    (8, 8, 4, 64, 100, False),  # rows whole: a launch for the heads
]


def close(got, want, bound, what):
    assert got.shape == want.shape
    assert np.abs(got - want).max() <= bound, what


@pytest.mark.parametrize("B,kvh,rep,hd,T,segments", STEPS)
def test_heads_finished_by_attention(B, kvh, rep, hd, T, segments):
    be = backend_with_env(**({"CG_ATTN_SEG_FROM": "1"} if segments else {}))
    H, rng = kvh * rep, np.random.default_rng(T + hd)
    r = lambda *s: rng.standard_normal(s).astype(np.float32)  # noqa: E731
    w = [r(n * hd, K) / np.float32(K ** 0.5) for n in (H, kvh, kvh)]
    gains = [1 + 0.3 * r(hd) for _ in range(2)]
    caches = [r(B, kvh, T, hd), r(B, kvh, T, hd)]
    angle = rng.uniform(0, 6.28, (T + 2, hd)).astype(np.float32)
    tables = [np.cos(angle), np.sin(angle)]
    tw, tg, tt, (tk, tv) = ([be.from_numpy(a) for a in group] for group in (w, gains, tables, caches))
    ck, cv = (c.astype(np.float64) for c in caches)
    for pos in (T, T + 1):
        x = r(B, 1, K)
        tx = be.from_numpy(x)
        q, k, v = (cases._linear(be, tx, a) for a in tw)

        def finish(t, n, gain):
            flat = be.reshape(be.transpose(be.reshape(t.move(), (B, 1, n, hd)).move(), 1, 2).move(), (B * n, hd))
            y = be.reshape(cases._rmsnorm_ops(be, flat, gain, hd, (B * n, hd)).move(), (B, n, 1, hd))
            del flat
            c, s = (be.broadcast(be.reshape(be.slice(a, 0, pos, 1).move(), (1, 1, 1, hd)).move(), (B, n, 1, hd)) for a in tt)
            mixed = cases._rot_half(be, y, hd // 2)
            return be.add(be.mul(c.move(), y.move()).move(), be.mul(s.move(), mixed.move()).move())

        q, k = finish(q, H, tg[0].clone()), finish(k, kvh, tg[1].clone())
        v = be.transpose(be.reshape(v.move(), (B, 1, kvh, hd)).move(), 1, 2)
        tk, tv = be.concat(tk.move(), k.move(), 2), be.concat(tv.move(), v.move(), 2)
        held = q.clone()
        out = be.to_numpy(cases.decode_attention_ops(be, q, tk.clone(), tv.clone(), rep))

        def head(a, n, gain):
            y = (x[:, 0].astype(np.float64) @ a.T.astype(np.float64)).reshape(B, n, hd)
            y = y / np.sqrt((y * y).mean(-1, keepdims=True) + EPS) * gain
            return y * tables[0][pos] + np.concatenate([-y[..., hd // 2:], y[..., :hd // 2]], -1) * tables[1][pos]

        wq, wk = head(w[0], H, gains[0]), head(w[1], kvh, gains[1])
        wv = (x[:, 0].astype(np.float64) @ w[2].T.astype(np.float64)).reshape(B, kvh, hd)
        ck, cv = np.concatenate([ck, wk[:, :, None]], 2), np.concatenate([cv, wv[:, :, None]], 2)
        scores = np.einsum("bgrd,bgtd->bgrt", wq.reshape(B, kvh, rep, hd), ck) / np.sqrt(hd)
        p = np.exp(scores - scores.max(-1, keepdims=True))
        p /= p.sum(-1, keepdims=True)
        want = np.einsum("bgrt,bgtd->bgrd", p, cv).reshape(B, H, 1, hd)
        # a value of q or k is off by sqrt(K) 2^-24 of its scale in the mean (2 to spare: the norm's sum, its division, the embedding), a score
        # by that much of |q| |k|, and what it weighs by as much of the largest value; the largest of the errors is taken as four times the mean
        u = 4 * 2 * K ** 0.5 * 2.0 ** -24
        length = np.linalg.norm(wq, axis=-1).max() * np.linalg.norm(ck, axis=-1).max() / np.sqrt(hd)
        close(be.to_numpy(held)[:, :, 0], wq, u * np.abs(wq).max(), "q")
        close(be.to_numpy(be.slice(tk, 2, 0, pos + 1)), ck, u * np.abs(ck).max(), "K")
        close(out, want, u * (length + T ** 0.5) * np.abs(cv).max(), "attention")
    del tw, tg, tt, tk, tv, tx, q, k, v, held
    be.close()
