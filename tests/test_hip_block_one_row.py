"""The decoder blocks' products of one row: shares of k that end inside a lane's values or leave waves without any, several trips, both
weight formats, operands in two parts, norms, gates and the polynomial norm, against float64."""
import numpy as np
import pytest

import block_cases as C
import loretar_reference as R

pytestmark = pytest.mark.gpu


def bound(x, w, k):  # a rounding per value of k in a lane and per addition of the lanes' and waves' sums, relative to the sum of magnitudes
    return (k / 64 + 32) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T)


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("K", [136, 264, 512, 520, 1024, 1032, 2048, 2056, 3072, 4096, 4104, 6144, 8192])
def test_linear(hip, K, dt):
    rng = np.random.default_rng(K)
    N, K1 = 1021, K // 16 * 8
    x, gamma, bias = rng.standard_normal((1, 1, K)).astype(np.float32), rng.uniform(0.5, 1.5, K).astype(np.float32), rng.standard_normal(N).astype(np.float32)
    w = C.bf16(rng.standard_normal((N, K)) * K ** -0.5)
    tw, f = C.weight(hip, w, dt), x[0, 0].astype(np.float64)
    parts = hip.from_numpy(x[:, :, :K1]), hip.from_numpy(x[:, :, K1:])
    got = hip.to_numpy(hip.block_linear(parts[0], tw, x2=parts[1], bias=hip.from_numpy(bias), scale=1.5))[0, 0]
    # (beside bfloat16 weights activations may be rounded to bfloat16)
    each = 0.0 if dt == "f32" else 2.0 ** -8
    b = bound(f, w, K) + each * (np.abs(f) @ np.abs(w).T)
    assert (np.abs(got - (1.5 * (w.astype(np.float64) @ f) + bias)) <= 2 * b + 2.0 ** -22 * np.abs(bias)).all()
    got = hip.to_numpy(hip.block_linear(hip.from_numpy(x), tw, gamma=hip.from_numpy(gamma), eps=1e-3))[0, 0]
    y = R.rms_norm(f[None], gamma.astype(np.float64), 1e-3)[0]
    assert (np.abs(got - w.astype(np.float64) @ y) <= bound(y, w, K) + (each + 2.0 ** -20) * (np.abs(y) @ np.abs(w).T)).all()


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("parts", [
    [(8, False, True), (24, True, True)], [(2048, False, True), (3072, True, True)], [(1024, False, False), (1032, False, True)], [(2056, False, True), (8192, True, True)],
    [(4104, True, False)], [(4096, False, True)], [(6144, False, True), (512, True, False)], [(16384, False, True)], [(8200, True, True)]])
def test_residual(hip, parts, dt):
    for width in (130, 1025):
        C.run_residual(hip, (1, width, parts, dt))
