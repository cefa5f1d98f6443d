"""h + x W^T for a few rows with the sum in the product's store: eight columns per workgroup and all of K by its eight waves."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 3, 4])
@pytest.mark.parametrize("K", [2048, 4096, 8192, 6144, 2052])
@pytest.mark.parametrize("N", [2048, 2050, 2060, 512])
def test_sum_in_the_store(hip, rows, K, N):
    rng = np.random.default_rng(K + N + rows)
    x, w, h = (rng.standard_normal(s, dtype=np.float32) for s in ((rows, 1, K), (N, K), (rows, 1, N)))
    tx, th, tw = hip.from_numpy(x), hip.from_numpy(h), hip.from_numpy(w)
    y = hip.matmul(tx.move(), hip.broadcast(hip.transpose(tw, 0, 1), (rows, K, N)).move())
    got = hip.to_numpy(hip.add(th, y.move()))[:, 0]
    a, b = x[:, 0].astype(np.float64), w.T.astype(np.float64)
    # a rounding per value of k and per addition of the partial sums, relative to the sum of magnitudes
    bound = (K + 64) * 2.0 ** -24 * (np.abs(a) @ np.abs(b)) + 2.0 ** -23 * np.abs(h[:, 0])
    assert (np.abs(got - (h[:, 0] + a @ b)) <= bound).all()
