"""The tokens' own vectors end in a sum of rows; filters over what it leaves take it into their launch for one token per sequence, and
whatever else comes next launches it first.  The results are those of separate launches, to the bit (test_hip_blocks.py has both
against the reference)."""
import numpy as np
import pytest

import block_cases as C
import kernel_names

pytestmark = pytest.mark.gpu

# sequences, width, groups, taps, outputs, whether there is a state: one to three pieces of a workgroup's loads, a group in two workgroups, groups shorter than a wave's piece and
# longer than one; other numbers of taps, a width that is not whole 16-byte pieces (neither goes along)
SHARES = [True] * 7 + [False] * 2
CASES = [(1, 1024, 4, 4, 2, True), (3, 1024, 1, 4, 2, True), (2, 2048, 8, 4, 1, False), (1, 2304, 1, 4, 2, True), (8, 264, 2, 4, 1, True), (1, 96, 3, 4, 2, False), (1, 4096, 2, 4, 2, True),
         (2, 1024, 4, 3, 2, True), (1, 262, 2, 4, 1, True)]


def run(be, case, between, dt="bf16", S=1):
    B, W, groups, taps, n, has_state = case
    rng = np.random.default_rng(W + B)
    dim, vocab = 128, 60
    x, table = rng.standard_normal((B, S, W)).astype(np.float32), C.bf16(rng.standard_normal((vocab, 4 * dim)))
    ids = rng.integers(0, vocab, size=(B, S), dtype=np.uint32)
    gate, proj = C.bf16(rng.standard_normal((dim, W)) * W ** -0.5), C.bf16(rng.standard_normal((W, dim)) * dim ** -0.5)
    norm = (1 + 0.3 * rng.standard_normal(W)).astype(np.float32)
    side = {"x": be.from_numpy(x), "ids": be.from_numpy(ids), "table": C.weight(be, table, dt), "gate": C.weight(be, gate, dt), "proj": C.weight(be, proj, dt), "norm": be.from_numpy(norm)}
    f = lambda *s: be.from_numpy(rng.standard_normal(s).astype(np.float32))
    ins = [{"gamma": f(W), "conv": f(W, taps), "w": C.weight(be, C.bf16(rng.standard_normal((40, W)) * W ** -0.5), dt), "keep": 1} for _ in range(n)]
    state = f(B, taps - 1, W) if has_state else be.zeros((B, taps - 1, W), 0)
    for t in list(side.values()) + [d[k] for d in ins for k in ("gamma", "conv", "w")] + ([state] if has_state else []):
        be.realize(t)
    small = [{k: (v.move() if k != "keep" else v) for k, v in d.items()} for d in ins]
    z = be.block_token_side({k: v.move() for k, v in side.items()}, first=dim, eps=2e-3, scale=0.6)
    kept = between(be, z)
    y, h, s = be.block_conv_linear(z, state, small, groups=groups, eps=2e-3)
    return [be.to_numpy(t) for t in [z, s] + y + [be.cast(t, 0) for t in h]] + ([] if kept is None else [be.to_numpy(t) for t in kept])


def same(a, b):
    for p, q in zip(a, b):
        np.testing.assert_array_equal(p, q)


@pytest.mark.parametrize("case", CASES, ids=str)
@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_same_results(hip, case, dt):
    same(run(hip, case, lambda be, z: None, dt), run(hip, case, lambda be, z: be.sync(), dt))


def test_two_tokens(hip):
    same(run(hip, CASES[0], lambda be, z: None, S=2), run(hip, CASES[0], lambda be, z: be.sync(), S=2))


def reads_result(be, z):
    return [be.add(z, z)]


def drops_memory(be, z):
    be.pool_trim()
    return [be.from_numpy(np.full((300, 300), 2.0, dtype=np.float32))]


def another_sum(be, z):
    return [be.block_residual(z, [], scale=1.0)]


@pytest.mark.parametrize("between", [reads_result, drops_memory, another_sum], ids=lambda f: f.__name__)
def test_what_else_comes_next(hip, between):
    same(run(hip, CASES[0], between), run(hip, CASES[0], lambda be, z: (be.sync(), between(be, z))[1]))


def test_filters_over_something_else(hip):
    """The rows that are filtered are others, and the sum's are their state or their gains: it comes first."""
    def as_operands(be, z):
        W = z.shape[-1]
        other, w = be.from_numpy(np.linspace(-1, 1, W, dtype=np.float32).reshape(1, 1, W)), be.from_numpy(np.eye(8, W, dtype=np.float32))
        conv = be.from_numpy(np.full((W, 2), 0.25, dtype=np.float32))
        y, h, s = be.block_conv_linear(other, z, [{"gamma": be.reshape(z, (W,)), "conv": conv, "w": w, "keep": 1}], groups=2, eps=1e-3)
        return y + h + [s]
    same(run(hip, CASES[0], as_operands), run(hip, CASES[0], lambda be, z: (be.sync(), as_operands(be, z))[1]))


def test_result_dropped(hip):
    run(hip, CASES[0], lambda be, z: None)
    before = hip.pool_stats()[0]
    for _ in range(3):
        run(hip, CASES[0], lambda be, z: None)
    hip.sync()
    assert hip.pool_stats()[0] <= before + 4096


def test_which_share(tmp_path):
    """The filters take the sum along where they should, and it runs by itself everywhere else."""
    kernel_names.run(tmp_path, r"""
from catgrad_amd import HipBackend
import test_hip_shared_sum as T
be = HipBackend(0)


def check(what, shares, *a, **kw):
    names = launches(be, T.run, be, *a, **kw)
    own = sum("side_sum_kernel" in k for k in names)
    print(what, own, flush=True)
    assert own == 1 - shares, names
    assert sum("conv_token_kernelILb1E" in k or "conv_token_kernel<true>" in k for k in names) == shares, names


for case, shares in zip(T.CASES, T.SHARES):
    check(case, int(shares), case, lambda be, z: None)
    check("with a wait", 0, case, lambda be, z: be.sync())
check("two tokens", 0, T.CASES[0], lambda be, z: None, S=2)
for f in (T.reads_result, T.drops_memory, T.another_sum):
    check(f.__name__, 0, T.CASES[0], f)
print("done", flush=True)
""")
