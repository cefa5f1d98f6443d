"""Products of operands that lie in memory as bfloat16, binary16 or fp8 patterns, on 128-wide tiles (cut along k or not) and at the
edges of the 256-wide ones: the sum in 32 bits, rounded once to the dtype."""
import numpy as np
import pytest

from catgrad_amd import _abi as A

pytestmark = pytest.mark.gpu

UNIT = {"bf16": 2.0 ** -8, "f16": 2.0 ** -11, "fp8": 2.0 ** -4}   # largest relative rounding error
# edges of tiles (64 / 128 rows, 128 columns), of stages (64 bytes of k), cuts along k, one column, odd results
SIZES = [(9, 16, 640), (64, 512, 129), (65, 272, 1021), (130, 1040, 520), (300, 2048, 260), (513, 192, 128), (1100, 64, 72), (4100, 2048, 16)]
WIDE = [("bf16", 1500, 256, 5632), ("f16", 1100, 128, 6660), ("fp8", 2100, 256, 8196)]   # whole turns of k, ragged rows and columns


def backend_values(be, torch, name, x):
    code, dt, bits, make = {"bf16": (A.BF16, torch.bfloat16, torch.int16, lambda r, s: be.ndarray_from_vec_bf16(r.view(np.uint16), s)),
                            "f16": (A.F16, torch.float16, torch.int16, lambda r, s: be.ndarray_from_vec_f16(r.view(np.float16), s)),
                            "fp8": (A.F8, torch.float8_e4m3fn, torch.uint8, be.ndarray_from_vec_fp8)}[name]
    t = torch.from_numpy(x).to(dt)
    return make(t.view(bits).numpy().reshape(-1), x.shape), t.double().numpy()


def run(be, name, M, K, N):
    import torch

    rng = np.random.default_rng(M + K + N)
    x, a = backend_values(be, torch, name, rng.standard_normal((1, M, K), dtype=np.float32))
    w, b = backend_values(be, torch, name, rng.standard_normal((N, K), dtype=np.float32) * np.float32(K ** -0.5))
    got = be.to_numpy(be.cast(be.matmul(x, be.broadcast(be.transpose(w, 0, 1), (1, K, N))), A.F32))[0]
    want = a[0].astype(np.float32) @ b.T.astype(np.float32) if M * N * K > 1 << 31 else a[0] @ b.T
    # the rounding to the dtype (fp8 below 2^-6: in steps of 2^-9) and the 32-bit sums of both sides
    bound = UNIT[name] * np.abs(want) + (2.0 ** -10 if name == "fp8" else 2.0 ** -25) + 2 * K * 2.0 ** -24 * 8.0
    assert (np.abs(got - want) <= bound).all()


@pytest.mark.parametrize("name", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("size", SIZES, ids=str)
def test_against_float64(hip, name, size):
    run(hip, name, *size)


@pytest.mark.parametrize("case", WIDE, ids=str)
def test_edges_of_the_wide_tile(hip, case):
    run(hip, *case)


def test_fp8_sums_keep_32_bits(hip):
    """Sums that lie within 2^-20 of the middle between two fp8 values go to the right one."""
    import torch

    M, K, N = 80, 4096, 640
    x = np.zeros((1, M, K), dtype=np.float32)
    w = np.zeros((N, K), dtype=np.float32)
    x[0, :, 0], w[:, 0] = 16.0, 1.0
    x[0, :, 1], w[:, 1] = 1.0, 1.0                # half way between 16 and 18, and 16 is even
    x[0, :, 2], w[:, 2] = 2.0 ** -6, 2.0 ** -9    # a push upwards
    xs, _ = backend_values(hip, torch, "fp8", x)
    ws, _ = backend_values(hip, torch, "fp8", w)
    got = hip.to_numpy(hip.cast(hip.matmul(xs, hip.broadcast(hip.transpose(ws, 0, 1), (1, K, N))), A.F32))
    assert (got == 18.0).all()                    # 16 + 1 + 2^-15


@pytest.mark.parametrize("M", [40, 200])
def test_fp8_results_at_the_ends_of_the_range(hip, M):
    """Sums beyond the largest value are that value, NaN stays NaN, small ones round to multiples of 2^-9."""
    import torch

    K, N = 256, 1024
    rng = np.random.default_rng(M)
    x = rng.standard_normal((1, M, K), dtype=np.float32)
    x[0, ::3] *= 100.0
    x[0, 1::3] = np.where(np.arange(K) < 2, rng.integers(-8, 9, (len(x[0, 1::3]), K)) * 2.0 ** -9, 0.0)
    x[0, 5, 7] = np.nan
    w = np.where(np.arange(K) < 2, 0.5, rng.standard_normal((N, K))).astype(np.float32)
    xs, a = backend_values(hip, torch, "fp8", x)
    ws, b = backend_values(hip, torch, "fp8", w)
    got = hip.to_numpy(hip.cast(hip.matmul(xs, hip.broadcast(hip.transpose(ws, 0, 1), (1, K, N))), A.F32))[0]
    exact = a[0] @ b.T
    want = torch.from_numpy(np.clip(exact, -448, 448)).float().to(torch.float8_e4m3fn).float().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isnan(got[5]).all()
    small = np.arange(M) % 3 == 1
    np.testing.assert_array_equal(got[small & (np.arange(M) != 5)], want[small & (np.arange(M) != 5)])    # sums of two multiples of 2^-10: exact
    far = np.abs(exact) > 500
    assert far.sum() > 100 and (got[far] == 448 * np.sign(exact[far])).all()
    # everything from 448 up is 448; below, one rounding to the dtype of a sum of 256 roundings of at most 448 * 2^-24 each
    near, keep = np.clip(exact, -448, 448), ~np.isnan(want)
    assert (np.abs(got - near)[keep] <= UNIT["fp8"] * np.abs(near[keep]) + 2.0 ** -10 + 2 * K * 2.0 ** -24 * 448).all()


@pytest.mark.parametrize("dtype", [A.BF16, A.F16])
@pytest.mark.parametrize("shape", [(1024, 16484, 256), (1024, 16387, 128), (1030, 13412, 384), (2048, 8448, 1280), (8192, 2052, 128), (300, 65600, 128), (66600, 200, 128), (66600, 500, 128)])
def test_columns_left_over_by_the_rounds_of_wide_tiles(hip, dtype, shape):
    """Results whose last few 256-wide tiles would be a round of their own: those columns come from the 128-wide tiles, beside the others in
    the same rows (rounded in the store, or as words where a row is no whole number of fours), cut along k or not."""
    import torch

    M, N, K = shape
    rng = np.random.default_rng(M + N + K)
    x, w = (torch.from_numpy(rng.standard_normal(s, dtype=np.float32)) for s in ((M, K), (N, K)))
    kind = torch.bfloat16 if dtype == A.BF16 else torch.float16
    x, w = x.to(kind), w.to(kind)

    def up(t):
        if dtype == A.BF16:
            return hip.ndarray_from_vec_bf16(t.view(torch.int16).numpy().view(np.uint16), tuple(t.shape))
        return hip.ndarray_from_vec_f16(t.view(torch.int16).numpy().view(np.float16), tuple(t.shape))

    tx, tw = hip.reshape(up(x).move(), (1, M, K)), up(w)
    y = hip.matmul(tx, hip.broadcast(hip.transpose(tw, 0, 1), (1, K, N)).move())
    got = hip.to_numpy(hip.cast(y.move(), A.F32))[0]
    want = (x.cuda().float() @ w.cuda().float().T).cpu().numpy()
    # the result's rounding, and the sums' in 32 bits
    unit = 2.0 ** -8 if dtype == A.BF16 else 2.0 ** -11
    assert (np.abs(got - want) <= unit * np.abs(want) + 1e-5 * K ** 0.5).all()
