"""The kernels of one to eight rows of activations by name: with the RMS norm in their loads, which a norm has to be left open for, with eight
columns a workgroup at their edges, and products that share their launch with no other."""
import numpy as np
import pytest

import kernel_names
import test_hip_skinny as whole
from test_hip_skinny import KS, constant, linear

pytestmark = pytest.mark.gpu


def norm_of(hip, x, gamma, power, eps):
    """x / pow(sum(x x) / n + eps, e) * gamma, every handle given away at its last use: so the norm is left to the products that read it."""
    _, rows, K = x.shape
    h, row = hip.from_numpy(x), (1, rows, 1)
    s = hip.div(hip.sum(hip.mul(h, h).move()).move(), constant(hip, float(K), row).move())
    d = hip.pow(hip.add(s.move(), constant(hip, eps, row).move()).move(), constant(hip, power, row).move())
    return hip.mul(hip.div(h, hip.broadcast(d.move(), x.shape).move()).move(), hip.broadcast(gamma, x.shape).move())


@pytest.mark.parametrize("power,eps", [(0.5, 1e-5), (0.25, 1e-5), (0.5, 0.0)])
@pytest.mark.parametrize("rows", [1, 2, 4, 7])
@pytest.mark.parametrize("K", KS)
def test_norm_left_to_the_products(hip, K, rows, power, eps):
    """x / pow(sum(x x) / n + eps, e) * gamma in front of one product, of three and of a gated pair."""
    rng = np.random.default_rng(K + 1)
    N = 514
    x, gamma = rng.standard_normal((1, rows, K), dtype=np.float32), rng.uniform(0.5, 1.5, K).astype(np.float32)
    w = rng.standard_normal((3, N, K), dtype=np.float32) * np.float32(K ** -0.5)
    tg, tw = hip.from_numpy(gamma), [hip.from_numpy(a) for a in w]

    def normed():
        return norm_of(hip, x, tg, power, eps)

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


@pytest.mark.parametrize("K", [5120, 5124, 6140, 6144, 6148])
def test_one_row_in_three_trips(hip, K):
    """Eight waves of one row share up to 6144 values of k in three trips (4100 is among the others' sizes)."""
    whole.test_whole_numbers(hip, K, 1)
    test_norm_left_to_the_products(hip, K, 1, 0.5, 1e-5)


@pytest.mark.parametrize("rows", [2, 3, 5, 8])
@pytest.mark.parametrize("K", [1020, 1028, 2048, 2052, 4100])
def test_eight_columns(hip, K, rows):
    """Products of at least 8192 columns share the rows among eight: their last workgroup's columns, alone, in pairs and behind a norm."""
    rng = np.random.default_rng(K + rows)
    x = rng.integers(-3, 4, (1, rows, K)).astype(np.float32)
    for N in (8193, 8199):
        w = [rng.integers(-3, 4, (n, K)).astype(np.float32) for n in (N, 8192)]
        tx, tw = hip.from_numpy(x), [hip.from_numpy(a) for a in w]
        np.testing.assert_array_equal(hip.to_numpy(linear(hip, tx, tw[0]))[0], x[0] @ w[0].T)
        for y, a in zip([linear(hip, tx, t) for t in tw], w):
            np.testing.assert_array_equal(hip.to_numpy(y)[0], x[0] @ a.T)
        gamma = rng.uniform(0.5, 1.5, K).astype(np.float32)
        got = hip.to_numpy(linear(hip, norm_of(hip, x, hip.from_numpy(gamma), 0.5, 1e-5), tw[0]))[0]
        f = x[0].astype(np.float64)
        y = f / np.sqrt(np.mean(f * f, -1, keepdims=True) + 1e-5) * gamma
        assert (np.abs(got - y @ w[0].astype(np.float64).T) <= (K / 16 + 64) * 2.0 ** -24 * (np.abs(y) @ np.abs(w[0]).T)).all()


# rows, K, columns of a product alone, and whether it is worth these kernels (enough of the lanes busy for its rows and columns)
ALONE = [(1, 576, 2050, True), (1, 572, 2050, False), (1, 1028, 16384, False), (1, 4100, 2050, True), (1, 6148, 2050, True), (1, 8196, 2050, False), (1, 956, 16384, True),
         (2, 1024, 2050, True), (2, 1028, 2050, False), (2, 2052, 2050, True), (2, 260, 16384, True), (2, 260, 16380, False),
         (4, 576, 2050, True), (4, 572, 2050, False), (3, 3580, 2050, False), (3, 3584, 2050, True), (4, 4100, 2050, True), (4, 2812, 16384, False), (4, 2816, 16384, True), (3, 260, 16384, True),
         (8, 2048, 2050, True), (5, 2052, 2050, False), (5, 2304, 8188, True), (8, 2560, 2050, True), (6, 3324, 8192, False), (5, 3328, 8192, True), (7, 2304, 8192, True), (7, 2300, 8192, False), (8, 6148, 8194, True),
         (8, 764, 16384, False), (8, 768, 16384, True), (5, 3836, 16384, False), (5, 3840, 16384, True), (8, 6148, 16384, True)]


def alone(hip, rows, K, N):
    rng = np.random.default_rng(K)
    x, w = rng.integers(-3, 4, (1, rows, K)).astype(np.float32), rng.integers(-3, 4, (N, K)).astype(np.float32)
    np.testing.assert_array_equal(hip.to_numpy(linear(hip, hip.from_numpy(x), hip.from_numpy(w)))[0], x[0] @ w.T)


def test_which_kernels(tmp_path):
    """The kernels with the norm in their loads run where it stands in front of the products, eight columns where there are enough, and a
    product alone goes where the rule says."""
    kernel_names.run(tmp_path, r"""
import re
from catgrad_amd import HipBackend
import test_hip_skinny_norms as T
be = HipBackend(0)


def count(names, pattern):
    return sum(bool(re.search(pattern, n)) for n in names)


for rows, K in ((1, 260), (1, 4100), (2, 1024), (4, 3084), (7, 8196)):
    names = launches(be, T.test_norm_left_to_the_products, be, K, rows, 0.5, 1e-5)
    print("norm", rows, K, flush=True)
    # (one product, three, and the gated pair, each with the norm in its loads)
    assert count(names, r"skinny_group_kernel.*Li4ELb1EE") == 2 and count(names, r"skinny_gated_kernel.*Lb1EE") == 1 and not count(names, "fused"), names
    names = launches(be, T.whole.test_whole_numbers, be, K, rows)
    # (three widths: a group of three, a residual sum; the products alone are below)
    assert count(names, r"skinny_group_kernel.*Li4ELb0EE") >= 3 and count(names, "skinny_residual_kernel") == 3, names
for rows, K in ((2, 1028), (8, 2052)):
    names = launches(be, T.test_eight_columns, be, K, rows)
    print("eight", rows, K, flush=True)
    assert count(names, r"skinny_group_kernel.*Li8ELb1EE") == 2 and count(names, r"skinny_group_kernel.*Li8ELb0EE") == 2, names
for rows, K, N, there in T.ALONE:
    names = launches(be, T.alone, be, rows, K, N)
    print("alone", rows, K, N, flush=True)
    assert count(names, "skinny_group_kernel") == there, names
print("done", flush=True)
""")
