"""Decode-time attention that norms and embeds the heads of q and of the cache's newest row itself, on every kernel that can and beside those that
leave it to a launch of its own, against float64: a step that appends by copying the caches (whose copies a launch for the heads comes before)
and one that appends in place.  Where the values are K's own cache, that launch has to store the newest row before attention asks for it."""
import numpy as np
import pytest

import cases
import kernel_names
from backends import backend_with_env

pytestmark = pytest.mark.gpu

K, EPS = 516, 1e-5
# (sequences, KV heads, query heads a KV head, head size, cached positions, always in segments)
ROWS = [  # a row a workgroup
    (1, 8, 2, 128, 1, False), (1, 8, 2, 128, 159, False), (1, 8, 2, 128, 160, False), (3, 2, 2, 128, 319, False), (1, 8, 2, 128, 470, False),
    (1, 3, 3, 64, 320, False), (2, 3, 1, 64, 640, False), (1, 3, 3, 64, 960, False), (2, 1, 8, 64, 1100, False),
    (3, 3, 1, 64, 4099, False),  # ... in two segments
]
SEGMENTS = [
    (1, 8, 2, 128, 1030, False), (4, 8, 2, 128, 700, False), (1, 3, 3, 64, 1024, True), (2, 1, 6, 64, 1023, True), (2, 1, 8, 128, 1025, True),
    (8, 8, 2, 128, 700, True), (8, 8, 3, 64, 1030, True),  # ... of several trips
]
APART = [(8, 8, 4, 64, 100, False), (8, 8, 5, 64, 1030, True)]  # rows whole, more values than wait for company: a launch for the heads
PROGRAMS = [(1, 1, 8, 128, 600, False), (1, 1, 8, 64, 1100, False), (1, 1, 6, 64, 1023, True)]  # one row of keys: its norm is not left open
# ... with one cache for K and V
SHARED = [(1, 8, 2, 128, 160, False), (1, 3, 3, 64, 320, False), (3, 3, 1, 64, 4099, False), (1, 8, 2, 128, 1030, True), (1, 3, 3, 64, 1024, True), (8, 8, 3, 64, 1030, True)]


def close(got, want, bound, what):
    assert got.shape == want.shape
    assert np.abs(got - want).max() <= bound, what


def finish(be, t, shape, gain, tables, pos):
    """Heads of a product, normed and embedded."""
    B, n, hd = shape
    flat = be.reshape(be.transpose(be.reshape(t.move(), (B, 1, n, hd)).move(), 1, 2).move(), (B * n, hd))
    y = cases._rmsnorm_ops(be, flat, gain, hd, (B * n, hd))
    del flat  # (the norm stays open if nobody else holds the product)
    y = be.reshape(y.move(), (B, n, 1, hd))
    c, s = (be.broadcast(be.reshape(be.slice(a, 0, pos, 1).move(), (1, 1, 1, hd)).move(), (B, n, 1, hd)) for a in tables)
    mixed = cases._rot_half(be, y, hd // 2)
    return be.add(be.mul(c.move(), y.move()).move(), be.mul(s.move(), mixed.move()).move())


def run(B, kvh, rep, hd, T, segments, shared=False, between=lambda: None):
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
        between()
        x = r(B, 1, K)
        tx = be.from_numpy(x)
        q, k, v = (cases._linear(be, tx, a) for a in tw)
        q, k = finish(be, q, (B, H, hd), tg[0].clone(), tt, pos), finish(be, k, (B, kvh, hd), tg[1].clone(), tt, pos)
        v = be.transpose(be.reshape(v.move(), (B, 1, kvh, hd)).move(), 1, 2)
        tk = be.concat(tk.move(), k.move(), 2)
        if not shared:
            tv = be.concat(tv.move(), v.move(), 2)
        held = q.clone()
        out = be.to_numpy(cases.decode_attention_ops(be, q, tk.clone(), (tk if shared else tv).clone(), rep))

        def head(a, n, gain):
            y = (x[:, 0].astype(np.float64) @ a.T.astype(np.float64)).reshape(B, n, hd)
            y = y / np.sqrt((y * y).mean(-1, keepdims=True) + EPS) * gain
            return y * tables[0][pos] + np.concatenate([-y[..., hd // 2:], y[..., :hd // 2]], -1) * tables[1][pos]

        wq, wk = head(w[0], H, gains[0]), head(w[1], kvh, gains[1])
        wv = (x[:, 0].astype(np.float64) @ w[2].T.astype(np.float64)).reshape(B, kvh, hd)
        ck = np.concatenate([ck, wk[:, :, None]], 2)
        cv = ck if shared else np.concatenate([cv, wv[:, :, None]], 2)
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


@pytest.mark.parametrize("B,kvh,rep,hd,T,segments", ROWS + SEGMENTS + APART + PROGRAMS)
def test_heads_finished_by_attention(B, kvh, rep, hd, T, segments):
    run(B, kvh, rep, hd, T, segments)


@pytest.mark.parametrize("B,kvh,rep,hd,T,segments", SHARED)
def test_one_cache_for_keys_and_values(B, kvh, rep, hd, T, segments):
    run(B, kvh, rep, hd, T, segments, shared=True)


def rows_of(T, hd, apart):
    """q and the newest row of K of a step behind T positions, from whole numbers; `apart`: over one cache, so that the heads get a launch of their own."""
    be = backend_with_env()
    B, kvh, rep = 2, 3, 2
    H, rng = kvh * rep, np.random.default_rng(hd)
    whole = lambda *s: rng.integers(-3, 4, s).astype(np.float32)  # noqa: E731
    tw = [be.from_numpy(whole(n * hd, K)) for n in (H, kvh, kvh)]
    gains = [be.from_numpy(rng.uniform(0.5, 1.5, hd).astype(np.float32)) for _ in range(2)]
    angle = rng.uniform(0, 6.28, (T + 2, hd)).astype(np.float32)
    tables = [be.from_numpy(f(angle)) for f in (np.cos, np.sin)]
    tk, tv = (be.from_numpy(whole(B, kvh, T, hd)) for _ in range(2))
    for pos in (T, T + 1):
        tx = be.from_numpy(whole(B, 1, K))
        q, k, v = (cases._linear(be, tx, a) for a in tw)
        q, k = finish(be, q, (B, H, hd), gains[0].clone(), tables, pos), finish(be, k, (B, kvh, hd), gains[1].clone(), tables, pos)
        v = be.transpose(be.reshape(v.move(), (B, 1, kvh, hd)).move(), 1, 2)
        tk, tv = be.concat(tk.move(), k.move(), 2), be.concat(tv.move(), v.move(), 2)
        held = q.clone()
        be.to_numpy(cases.decode_attention_ops(be, q, tk.clone(), (tk if apart else tv).clone(), rep))
    return [be.to_numpy(held), be.to_numpy(be.slice(tk, 2, T + 1, 1))]


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("T", [37, 300])
def test_rows_do_not_depend_on_the_launch(T, hd):
    """Sums of squares of whole numbers are exact in any order: all that follows them is the same to the bit."""
    for a, b in zip(rows_of(T, hd, False), rows_of(T, hd, True)):
        np.testing.assert_array_equal(a, b)


def test_which_kernels(tmp_path):
    """Attention finishes the heads of the step that appends in place, or one launch of its own does."""
    kernel_names.run(tmp_path, r"""
from catgrad_amd import HipBackend
import test_hip_heads_by_attention as T
be = HipBackend(0)
for steps, expected in ((T.ROWS, (0, 1, 0)), (T.SEGMENTS, (0, 0, 1)), (T.APART, (1, 0, 0)), (T.PROGRAMS, (0, 0, 0)), (T.SHARED, (1, 0, 0))):
    for step in steps:
        names = launches(be, T.run, *step, steps is T.SHARED, shim.names)
        own = sum("head_norm_rope_finish" in n for n in names)
        row, seg = (sum("decode_attention_%s_kernel" % k in n and "RawHeads" in n for n in names) for k in ("row", "seg"))
        print(step, own, row, seg, flush=True)
        assert (own, row, seg) == expected, names
for apart in (False, True):
    names = launches(be, T.rows_of, 300, 64, apart)
    assert sum("RawHeads" in n for n in names) == 1 - apart, names
print("done", flush=True)
""")
