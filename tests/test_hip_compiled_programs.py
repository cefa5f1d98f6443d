"""Compositions whose fused programs have kernels of their own give the bits that the program interpreter gives."""
import numpy as np
import pytest

from catgrad_amd import _abi as A

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def interpreter(hip):
    from backends import backend_with_env

    be = backend_with_env(CG_AOT="0")
    hip.own_programs, be.own_programs = (1, 0), (0, 1)  # programs launched: compiled, interpreted
    yield be
    be.close()


def realized(be, y):
    """y computed in its own dtype, with a compiled program (or, on the backend without them, an interpreted one): a cast behind the
    program would make it another."""
    be.program_stats()
    be.realize(y)
    assert be.program_stats() == be.own_programs
    return be.to_numpy(be.cast(y.move(), A.F32))


def silu_mul(be, dtype, shape, rng):
    g, u = (be.cast(be.from_numpy(rng.standard_normal(shape, dtype=np.float32) * np.float32(4)), dtype) for _ in range(2))
    be.realize(g), be.realize(u)
    one = be.broadcast(be.cast(be.ndarray_from_vec_f32([1.0], ()), dtype).move(), shape)
    e = be.exp(be.neg(g).move())
    e = be.div(g.move(), be.add(one.move(), e.move()).move())
    return [realized(be, be.mul(e.move(), u.move()))]


def row_programs(be, shape, rng):
    v = rng.standard_normal(shape, dtype=np.float32) * np.float32(30)
    v[0, :] = np.float32(-3.4028235e38)                # a masked row
    v[-1, 0] = np.inf
    x = be.from_numpy(v)
    m = be.max(x)
    be.realize(m)
    e = be.exp(be.sub(x, be.broadcast(m, shape).move()).move())
    lse = be.add(be.log(be.sum(e.move()).move()).move(), m)
    m2 = be.max(x)
    e2 = be.exp(be.sub(x, be.broadcast(m2, shape).move()).move())
    soft = be.div(e2, be.broadcast(be.sum(e2), shape).move())
    return [be.to_numpy(lse), be.to_numpy(soft)]


def bias_sigmoid(be, shape, rng):
    x, b = be.from_numpy(rng.standard_normal(shape, dtype=np.float32) * np.float32(9)), be.from_numpy(rng.standard_normal(shape[-1:], dtype=np.float32))
    one = be.broadcast(be.ndarray_from_vec_f32([1.0], ()), shape)
    e = be.exp(be.neg(be.add(x, be.broadcast(b, shape).move()).move()).move())
    return [be.to_numpy(be.div(one, be.add(one, e.move()).move()))]


CASES = {f"silu_{A.DTYPE_NAMES[d]}_{s}": (lambda be, rng, d=d, s=s: silu_mul(be, d, s, rng))
         for d in (A.BF16, A.F16, A.F8) for s in ((1, 3, 7), (1, 130, 513), (1, 300, 1024))}
CASES.update({f"rows_{s}": (lambda be, rng, s=s: row_programs(be, s, rng)) for s in ((3, 33), (5, 100), (9, 1000), (4, 4096), (2, 20001))})
CASES.update({f"sigmoid_{s}": (lambda be, rng, s=s: bias_sigmoid(be, s, rng)) for s in ((1, 2, 5), (1, 64, 512), (2, 33, 1027))})


@pytest.mark.parametrize("name", list(CASES))
def test_compiled_and_interpreted_agree(hip, interpreter, name):
    got, want = (CASES[name](be, np.random.default_rng(11)) for be in (hip, interpreter))
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)


def gating(be, dtype, gate, up):
    raw = {A.BF16: be.ndarray_from_vec_bf16, A.F8: be.ndarray_from_vec_fp8}[dtype]
    g, u = raw(gate, gate.shape), raw(up, up.shape)
    one = be.broadcast(be.cast(be.ndarray_from_vec_f32([1.0], ()), dtype).move(), gate.shape)
    e = be.exp(be.neg(g).move())
    e = be.div(g.move(), be.add(one.move(), e.move()).move())
    return realized(be, be.mul(e.move(), u.move()))


@pytest.mark.parametrize("extra", [0, 1, 7, 9, 15, 4097])
@pytest.mark.parametrize("dtype", [A.BF16, A.F8])
def test_gating_of_every_value(hip, interpreter, dtype, extra):
    """All patterns of the dtype as gates, beside several factors; counts that end inside a lane's share, a workgroup's, and beyond."""
    rng = np.random.default_rng(extra)
    bits, kind = (16, np.uint16) if dtype == A.BF16 else (8, np.uint8)
    # (large enough to lie in memory as patterns, not words; many whole rounds of the patterns in a run, so that fast and slow meet)
    gate = np.concatenate([np.arange(1 << bits, dtype=kind)] * max(2, (1 << 18) >> bits) + [rng.integers(0, 1 << bits, extra, dtype=kind)])
    up = rng.integers(0, 1 << bits, gate.size, dtype=kind)
    up[: 1 << bits] = {A.BF16: 0x3F80, A.F8: 0x38}[dtype]  # one
    got, want = (gating(be, dtype, gate, up) for be in (hip, interpreter))
    np.testing.assert_array_equal(got, want)
    small = rng.integers(0, 0x4281 if dtype == A.BF16 else 256, gate.size, dtype=kind)  # gates of the fast range alone, both signs
    if dtype == A.BF16:
        small |= (rng.integers(0, 2, gate.size, dtype=kind) << 15).astype(kind)
    got, want = (gating(be, dtype, small, up) for be in (hip, interpreter))
    np.testing.assert_array_equal(got, want)
    if dtype == A.BF16:
        every = np.concatenate([np.arange(0x4281, dtype=kind), np.arange(0x8000, 0xC281, dtype=kind)] * 8)
        ones = np.full(every.size, 0x3F80, kind)
        got, want = (gating(be, dtype, every, ones) for be in (hip, interpreter))
        np.testing.assert_array_equal(got, want)
