"""Attention over mixed scores of a few tokens shares its launch with the experts that come next; whatever else comes next launches it
first.  The results are those of separate launches, to the bit (test_hip_blocks.py has both against the reference)."""
import numpy as np
import pytest

import block_cases as C
import kernel_names

pytestmark = pytest.mark.gpu

# query heads per kv head and head widths that the shared kernel is compiled for, one that it is not (16 columns), a model's width in one to
# eight pieces of a wave's loads and beyond, rows whose length is not whole 16-byte pieces; LDS for two workgroups
SHARES = [True, True, True, True, True, True, False, False, False, False, True]
CASES = [(4, 4, 64, 64, 256, "f32", 1, 1), (8, 4, 128, 128, 1024, "f32", 1, 1), (8, 2, 48, 32, 520, "bf16", 1, 2), (16, 8, 128, 128, 1024, "bf16", 2, 2), (8, 2, 96, 64, 2048, "f32", 1, 8),
         (4, 2, 64, 64, 4096, "bf16", 1, 1), (4, 2, 64, 64, 4352, "f32", 1, 1), (4, 2, 64, 64, 262, "f32", 1, 1), (4, 2, 16, 16, 256, "f32", 1, 1), (16, 2, 64, 64, 256, "f32", 1, 1),
         (32, 8, 128, 64, 256, "f32", 1, 8)]


def run(be, case, between, seed=0):
    heads, kv_heads, dim, vdim, width, dt, B, S = case
    rng = np.random.default_rng(seed)
    o = C.turned(heads, kv_heads, dim, vdim, 16)
    cached, rows, count, ff = 70, B * S, 8, 24
    t = C.attention_case(rng, B, S, o, norms=False)
    cache = [be.from_numpy(rng.standard_normal((B, kv_heads, cached, d)).astype(np.float32)) for d in (dim, vdim)]
    e = C.expert_case(rng, rows, width, count, ff, dt)
    ex = {n: be.from_numpy(e[n].reshape((B, S, -1) if n == "logits" else e[n].shape)) for n in ("logits", "correction")}
    h = be.from_numpy(e["h"].reshape(B, S, width))
    ex["h"] = h if dt == "f32" else be.cast(h, C.BF16)
    ex.update({n: C.weight(be, e[n], dt) for n in ("gate_up", "down")})
    w = C.weight(be, C.bf16(rng.standard_normal((width, heads * vdim)) * (heads * vdim) ** -0.5), dt)
    x = be.from_numpy(rng.standard_normal((B, S, width)).astype(np.float32))
    for v in list(ex.values()) + [w, x]:
        be.realize(v)
    tensors = {n: be.from_numpy(t[n]) for n in ("q", "k", "v", "talk")}
    y, kc, vc = be.block_attention({**tensors, "k_cache": cache[0].move(), "v_cache": cache[1].move()}, position=cached, **o)
    kept = between(be, y, kc, vc, x)
    out = be.block_residual(x, [{"y": y.move() if kept is None else y, "w": w}], scale=0.4, experts=ex, top=2, groups=4, keep=2, limit=1.2, slope=1.702)
    res = [be.to_numpy(a) for a in (out, kc, vc)]
    return res + ([] if kept is None else [be.to_numpy(a) for a in kept])


def nothing(be, y, kc, vc, x):
    return None


def waits(be, y, kc, vc, x):
    be.sync()


@pytest.mark.parametrize("case", CASES, ids=str)
def test_same_results(hip, case):
    for a, b in zip(run(hip, case, nothing), run(hip, case, waits)):
        np.testing.assert_array_equal(a, b)


def reads_result(be, y, kc, vc, x):
    return [be.add(y, y)]


def reads_caches(be, y, kc, vc, x):
    return [be.add(kc, kc), be.add(vc, vc)]


def drops_memory(be, y, kc, vc, x):
    be.pool_trim()
    return [be.from_numpy(np.full((300, 300), 2.0, dtype=np.float32))]


@pytest.mark.parametrize("between", [reads_result, reads_caches, drops_memory], ids=lambda f: f.__name__)
def test_what_else_comes_next(hip, between):
    case = CASES[1]
    for a, b in zip(run(hip, case, between), run(hip, case, lambda *a: (waits(*a), between(*a))[1])):
        np.testing.assert_array_equal(a, b)


def test_a_residual_sum_of_something_else(hip):
    """The branch is not what attention leaves, and its other operands are: nothing is shared."""
    def other(be, y, kc, vc, x):
        n = y.shape[-1]
        w = be.from_numpy(np.eye(n, dtype=np.float32))
        z = be.block_residual(y, [{"y": y, "w": w}], scale=1.0)
        return [z, be.block_residual(x, [], scale=1.0)]
    case = CASES[1]
    got, want = run(hip, case, other), run(hip, case, lambda *a: (waits(*a), other(*a))[1])
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a, b)


def test_results_dropped(hip):
    before = hip.pool_stats()[0]
    heads, kv_heads, dim, vdim = 8, 4, 64, 64
    o = C.turned(heads, kv_heads, dim, vdim, 16)
    t = C.attention_case(np.random.default_rng(1), 1, 1, o, norms=False)
    for _ in range(3):
        caches = {n: hip.from_numpy(np.ones((1, kv_heads, 5, 64), dtype=np.float32)) for n in ("k_cache", "v_cache")}
        r = hip.block_attention({**{n: hip.from_numpy(t[n]) for n in t}, **caches}, position=5, **o)
        del r, caches
    hip.sync()
    assert hip.pool_stats()[0] <= before + 4096


def test_which_share(tmp_path):
    """The kernel that both share runs where it should, once, and nowhere else."""
    kernel_names.run(tmp_path, r"""
from catgrad_amd import HipBackend
import test_hip_shared_step as T
be = HipBackend(0)


def check(what, shares, *a):
    names = launches(be, T.run, be, *a)
    n = sum("attention_step_experts_kernel" in k for k in names)
    print(what, n, flush=True)
    assert n == shares and sum("attention_mixed_step_kernel" in k for k in names) == 1 - shares, names


for case, shares in zip(T.CASES, T.SHARES):
    check(case, int(shares), case, T.nothing)
    check("with a wait", 0, case, T.waits)
for f in (T.reads_result, T.reads_caches, T.drops_memory):
    check(f.__name__, 0, T.CASES[1], f)
print("done", flush=True)
""")
