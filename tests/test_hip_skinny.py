"""The linear layers of one to eight rows of activations (decode steps): products that share their left operand, gated pairs,
residual sums and RMS norms in the loads, at the edges of the waves' shares of k and of a workgroup's columns."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# every number of trips, whole and ragged; shares that end inside a quad of lanes' values; one and several rounds of 8192
KS = [260, 264, 1020, 1024, 1028, 2048, 2052, 3072, 3084, 4096, 4100, 8188, 8192, 8196, 16384, 16900]


def linear(hip, x, w):
    n, k = w.shape
    return hip.matmul(x, hip.broadcast(hip.transpose(w, 0, 1), (1, k, n)).move())


@pytest.mark.parametrize("rows", [1, 2, 3, 8])
@pytest.mark.parametrize("K", KS)
def test_whole_numbers(hip, K, rows):
    """Alone, as a group of columns that fill no workgroup, and in a residual sum: exact, whatever the order of summation."""
    rng = np.random.default_rng(K)
    x = rng.integers(-3, 4, (1, rows, K)).astype(np.float32)
    for N in (513, 2050, 4097):
        w = rng.integers(-3, 4, (3, N, K)).astype(np.float32)
        tx, tw = hip.from_numpy(x), [hip.from_numpy(a) for a in w]
        want = [x[0] @ a.T for a in w]
        np.testing.assert_array_equal(hip.to_numpy(linear(hip, tx, tw[0]))[0], want[0])
        for y, z in zip([linear(hip, tx, t) for t in tw], want):
            np.testing.assert_array_equal(hip.to_numpy(y)[0], z)
        r = rng.integers(-9, 10, (1, rows, N)).astype(np.float32)
        np.testing.assert_array_equal(hip.to_numpy(hip.add(linear(hip, tx, tw[1]).move(), hip.from_numpy(r)))[0], want[1] + r[0])


def constant(hip, v, shape):
    return hip.broadcast(hip.ndarray_from_vec_f32([v], ()), shape)


@pytest.mark.parametrize("power,eps", [(0.5, 1e-5), (0.25, 1e-5), (0.5, 0.0)])
@pytest.mark.parametrize("rows", [1, 2, 4, 7])
@pytest.mark.parametrize("K", KS)
def test_norm_and_gate(hip, K, rows, power, eps):
    """x / pow(sum(x x) / n + eps, e) * gamma in front of one product, of three and of a gated pair."""
    rng = np.random.default_rng(K + 1)
    N = 514
    x, gamma = rng.standard_normal((1, rows, K), dtype=np.float32), rng.uniform(0.5, 1.5, K).astype(np.float32)
    w = rng.standard_normal((3, N, K), dtype=np.float32) * np.float32(K ** -0.5)
    tg, tw = hip.from_numpy(gamma), [hip.from_numpy(a) for a in w]

    def normed():
        h = hip.from_numpy(x)
        row = (1, rows, 1)
        s = hip.div(hip.sum(hip.mul(h, h).move()).move(), constant(hip, float(K), row).move())
        d = hip.pow(hip.add(s.move(), constant(hip, eps, row).move()).move(), constant(hip, power, row).move())
        return hip.mul(hip.div(h, hip.broadcast(d, (1, rows, K)).move()).move(), hip.broadcast(tg, (1, rows, K)).move())

    f = x[0].astype(np.float64)
    y = f / (np.mean(f * f, -1, keepdims=True) + eps) ** power * gamma
    want = [y @ a.astype(np.float64).T for a in w]
    # a rounding per value of k and per sum of shares, and a handful of the norm's, relative to the sum of magnitudes
    bound = [(K / 16 + 64) * 2.0 ** -24 * (np.abs(y) @ np.abs(a).astype(np.float64).T) for a in w]
    n = normed()
    for got, z, b in zip([hip.to_numpy(linear(hip, n, t)) for t in tw[:1]] + [hip.to_numpy(p) for p in [linear(hip, n, t) for t in tw]], want[:1] + want, bound[:1] + bound):
        assert (np.abs(got[0] - z) <= b).all()
    n = normed()
    g, u = linear(hip, n, tw[0]), linear(hip, n, tw[1])
    e = hip.exp(hip.neg(g).move())
    one = constant(hip, 1.0, (1, rows, N))
    e = hip.div(one, hip.add(one, e.move()).move())
    got = hip.to_numpy(hip.mul(hip.mul(g.move(), e.move()).move(), u.move()))[0]
    s = want[0] / (1.0 + np.exp(-want[0]))
    # silu' <= 1.1; the sigmoid's own roundings
    assert (np.abs(got - s * want[1]) <= 1.1 * bound[0] * np.abs(want[1]) + np.abs(s) * bound[1] + 2.0 ** -20 * np.abs(s * want[1])).all()
