"""Compositions whose fused programs have kernels of their own give the bits that the program interpreter gives."""
import numpy as np
import pytest

from catgrad_amd import _abi as A

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def interpreter():
    from backends import backend_with_env

    be = backend_with_env(CG_AOT="0")
    yield be
    be.close()


def silu_mul(be, dtype, shape, rng):
    g, u = (be.cast(be.from_numpy(rng.standard_normal(shape, dtype=np.float32) * np.float32(4)), dtype) for _ in range(2))
    be.realize(g), be.realize(u)
    one = be.broadcast(be.cast(be.ndarray_from_vec_f32([1.0], ()), dtype).move(), shape)
    e = be.exp(be.neg(g).move())
    e = be.div(g.move(), be.add(one.move(), e.move()).move())
    return [be.to_numpy(be.cast(be.mul(e.move(), u.move()).move(), A.F32))]


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
