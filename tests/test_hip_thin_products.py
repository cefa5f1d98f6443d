"""Products of a few dozen rows with k contiguous in both operands, of f32 and of the narrow dtypes: a workgroup's waves take turns of
32 values (narrow: 128 bytes) of k, and their sums meet in LDS; f32 rows that the pieces cannot hold are multiplied as they are."""
import numpy as np
import pytest

from catgrad_amd import _abi as A

pytestmark = pytest.mark.gpu

# one value beside a block of 16 rows and columns, a turn (32 values of k), a round of turns (256) and the next waves' turns; more
# workgroups than compute units (two row blocks each); k that is not whole turns
SIZES = [(9, 8, 1), (16, 32, 16), (17, 28, 17), (16, 36, 15), (31, 256, 33), (33, 260, 16), (32, 516, 100), (48, 772, 65), (64, 1000, 48), (65, 1540, 17), (9, 2052, 31),
         (64, 1024, 4096), (30, 1028, 8192), (33, 100, 1000)]


def operands(be, M, K, N, batch=1, seed=0):
    rng = np.random.default_rng(seed)
    a, b = rng.standard_normal((batch, M, K), dtype=np.float32), rng.standard_normal((batch, N, K), dtype=np.float32)
    return a, b, be.from_numpy(a), be.transpose(be.from_numpy(b), 1, 2)


def check(got, a, b):
    a, b = a.astype(np.float64), b.astype(np.float64).transpose(0, 2, 1)
    # a wave's turns (every eighth of 32 values of k) with a rounding for each of the six kept products, then the eight waves' sums
    n = 6 * (((a.shape[-1] + 31) // 32 + 7) // 8) + 8
    want = a @ b
    # three left-out products of pieces (2^-24 together at most) and the roundings, each relative to the sum of magnitudes
    assert (np.abs(got - want) <= (1.0 + n) * 2.0 ** -24 * (np.abs(a) @ np.abs(b)) + 1e-37).all()
    # all of them together: roundings of either sign, of sums that are no larger than the results.  Stated in numpy, the six products come to
    # 0.09 to 0.23 of this, and to 4.4 and more where any one of the smaller five is left out.
    rms = lambda v: np.sqrt((v ** 2).mean())
    assert rms(got - want) <= (1.0 + np.sqrt(n)) * 2.0 ** -24 * rms(want)


@pytest.mark.parametrize("size", SIZES, ids=str)
def test_edges(hip, size):
    a, b, x, y = operands(hip, *size)
    check(hip.to_numpy(hip.matmul(x, y)), a, b)


def test_batches_and_views(hip):
    a, b, x, y = operands(hip, 40, 100, 90, batch=3)
    check(hip.to_numpy(hip.matmul(x, y)), a, b)
    x, y = hip.slice(x, 2, 4, 72), hip.slice(y, 1, 4, 72)
    check(hip.to_numpy(hip.matmul(x, y)), a[:, :, 4:76], b[:, :, 4:76])


@pytest.mark.parametrize("size", [(16, 96, 40), (40, 100, 130), (64, 1000, 48), (30, 1028, 8192)], ids=str)
@pytest.mark.parametrize("side", ["left", "right"])
def test_ends_of_the_range(hip, size, side):
    """Chosen by a unit matrix: rows of any magnitude come out as they are, beside infinities and NaN."""
    M, K, N = size
    rng = np.random.default_rng(M)
    rows = M if side == "left" else N
    a = np.ldexp(rng.standard_normal((rows, K)), rng.integers(-20, 20, (rows, K))).astype(np.float32)
    a[0] = np.float32(3.4028235e38) * np.sign(a[0])
    a[3] = np.ldexp(1 + rng.random(K), rng.integers(-149, -110, K)).astype(np.float32)
    a[5, ::2] = np.ldexp(1 + rng.random(len(a[5, ::2])), rng.integers(-149, 20, len(a[5, ::2]))).astype(np.float32)
    a[7, 1], a[8, 2] = np.inf, np.nan
    others = N if side == "left" else M
    at, b = rng.integers(0, K, others), np.zeros((others, K), dtype=np.float32)
    b[np.arange(others), at] = 1.0
    with np.errstate(all="ignore"):
        want = np.where((np.isfinite(a).sum(1)[:, None] - np.isfinite(a[:, at])) < K - 1, np.float32(np.nan), a[:, at])
    x, w = (a, b) if side == "left" else (b, a)
    got = hip.to_numpy(hip.matmul(hip.from_numpy(x), hip.transpose(hip.from_numpy(w), 0, 1)))
    np.testing.assert_array_equal(got if side == "left" else got.T, want)


@pytest.mark.parametrize("size", [(64, 1024, 1024), (32, 576, 1536), (64, 256, 512)], ids=str)
def test_roundings_have_no_direction(hip, size):
    """The error's mean over all results against their root mean square: below 2^-28 for roundings to nearest, 2^-27 and more for sums
    that are cut off below."""
    a, b, x, y = operands(hip, *size, seed=3)
    want = a.astype(np.float64) @ b.astype(np.float64).transpose(0, 2, 1)
    d = hip.to_numpy(hip.matmul(x, y)) - want
    assert abs(d.mean()) <= 2.0 ** -28 * np.sqrt((want ** 2).mean())


# a value beside a block of 16 rows and columns, a turn (64 16-bit or 128 8-bit values) and a round of the waves' turns; one and two row
# blocks per workgroup; a tall narrow result
NARROW = [(70, 1024, 65), (17, 4112, 17), (65, 1040, 128), (96, 1536, 600), (130, 560, 1500), (1500, 2048, 16), (64, 1008, 1000), (16, 8192, 100)]


@pytest.mark.parametrize("size", NARROW, ids=str)
@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float8"])
def test_narrow_dtypes(hip, size, dtype):
    """Exact sums of small whole numbers, so that the one rounding of the result is all there may be."""
    torch = pytest.importorskip("torch")
    M, K, N = size
    rng = np.random.default_rng(K)
    a, b = rng.integers(-3, 4, (M, K)).astype(np.float32), rng.integers(-3, 4, (N, K)).astype(np.float32)
    kind = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float8": torch.float8_e4m3fn}[dtype]
    make = {"bfloat16": lambda v: hip.ndarray_from_vec_bf16(torch.from_numpy(v).to(kind).view(torch.int16).numpy().view(np.uint16), v.shape),
            "float16": lambda v: hip.ndarray_from_vec_f16(v.astype(np.float16), v.shape),
            "float8": lambda v: hip.ndarray_from_vec_fp8(torch.from_numpy(v).to(kind).view(torch.uint8).numpy(), v.shape)}[dtype]
    got = hip.to_numpy(hip.cast(hip.matmul(make(a), hip.transpose(make(b), 0, 1)), A.F32))
    want = torch.from_numpy(a.astype(np.float64) @ b.astype(np.float64).T)
    want = (want.clamp(-448, 448) if dtype == "float8" else want).to(kind).float().numpy()
    np.testing.assert_array_equal(got, want)
