"""The decoder blocks' products of one row: shares of k that end inside a lane's values or leave waves without any, several trips, both
weight formats, operands in two parts, norms, gates and the polynomial norm, against float64."""
import numpy as np
import pytest

import block_cases as C
import kernel_names
import loretar_reference as R
from backends import backend_with_env

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def narrow():
    """Stores bfloat16 tensors of any size as such (others: from 65536 elements on)."""
    be = backend_with_env(CG_NARROW_FROM="2")
    yield be
    be.close()


def bound(x, w, k):  # a rounding per value of k in a lane and per addition of the lanes' and waves' sums, relative to the sum of magnitudes
    return (k / 64 + 32) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T)


KS = [136, 264, 512, 520, 1024, 1032, 2048, 2056, 3072, 4096, 4104, 6144, 8192]


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("K", KS)
def test_linear(narrow, K, dt):
    linear(narrow, K, dt)


def linear(hip, K, dt):
    rng = np.random.default_rng(K)
    N, K1 = 1021, K // 16 * 8
    x, gamma, bias = rng.standard_normal((1, 1, K)).astype(np.float32), rng.uniform(0.5, 1.5, K).astype(np.float32), rng.standard_normal(N).astype(np.float32)
    w = C.bf16(rng.standard_normal((N, K)) * K ** -0.5)
    tw, f = C.weight(hip, w, dt), x[0, 0].astype(np.float64)
    parts = hip.from_numpy(x[:, :, :K1]), hip.from_numpy(x[:, :, K1:])
    got = hip.to_numpy(hip.block_linear(parts[0], tw, x2=parts[1], bias=hip.from_numpy(bias), scale=1.5))[0, 0]
    # (activations stay in 32 bits, also beside bfloat16 weights, which are exact here)
    b = bound(f, w, K)
    assert (np.abs(got - (1.5 * (w.astype(np.float64) @ f) + bias)) <= 2 * b + 2.0 ** -22 * np.abs(bias)).all()
    got = hip.to_numpy(hip.block_linear(hip.from_numpy(x), tw, gamma=hip.from_numpy(gamma), eps=1e-3))[0, 0]
    y = R.rms_norm(f[None], gamma.astype(np.float64), 1e-3)[0]
    assert (np.abs(got - w.astype(np.float64) @ y) <= bound(y, w, K) + 2.0 ** -20 * (np.abs(y) @ np.abs(w).T)).all()


PARTS = [
    [(8, False, True), (24, True, True)], [(2048, False, True), (3072, True, True)], [(1024, False, False), (1032, False, True)], [(2056, False, True), (8192, True, True)],
    [(4104, True, False)], [(4096, False, True)], [(6144, False, True), (512, True, False)], [(16384, False, True)], [(8200, True, True)]]


def residual(be, parts, dt):
    for width in (130, 1025):
        C.run_residual(be, (1, width, parts, dt), behind=8)


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("parts", PARTS)
def test_residual(narrow, parts, dt):
    residual(narrow, parts, dt)


def test_which_kernels(tmp_path):
    """One row's kernels wherever a workgroup's registers hold its share of k (4096 values in 32 bits, 8192 in bfloat16; the sum: 8192, 16384)."""
    kernel_names.run(tmp_path, r"""
import test_hip_block_one_row_bounds as T
be = T.backend_with_env(CG_NARROW_FROM="2")
for dt in ("f32", "bf16"):
    for K in T.KS:
        n = sum("block_one_row_kernelILb%d" % (dt == "bf16") in k for k in launches(be, T.linear, be, K, dt))
        print(K, dt, n, flush=True)
        assert n == (2 if K <= (4096 if dt == "f32" else 8192) else 0)
    for parts in T.PARTS:
        n = sum("block_one_row_residual_kernelILb%d" % (dt == "bf16") in k for k in launches(be, T.residual, be, parts, dt))
        print(parts, dt, n, flush=True)
        assert n == (2 if max(p[0] for p in parts) <= (8192 if dt == "f32" else 16384) else 0)
print("done", flush=True)
""")
