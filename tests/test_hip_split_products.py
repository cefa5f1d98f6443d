"""f32 products of more than eight rows: multiplied in pieces of 8 significant bits, whatever the layout and wherever the tiles
end, to the accuracy of 32-bit arithmetic; rows that the pieces cannot hold are multiplied as they are."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# edges of the tiles (64 x 64, 32 x 256, 64 x 128, 128 x 128, 256 x 256), of a stage (16 values of k) and of the cuts along k
SIZES = [(9, 16, 8), (9, 1, 33), (17, 33, 31), (32, 2048, 260), (33, 96, 128), (64, 100, 129), (65, 576, 192), (128, 160, 256), (129, 31, 4), (255, 64, 260),
         (300, 1000, 520), (1030, 48, 1028), (2048, 64, 8192),
         (64, 64, 64), (65, 63, 65), (1800, 100, 400), (200, 1001, 333), (1500, 700, 50),
         (2048, 128, 8192), (1024, 64, 4096), (1030, 63, 4098), (20, 512, 8192)]


def operands(be, M, K, N, a_rows_fast, b_rows_fast, batch=1, seed=0):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((batch, M, K), dtype=np.float32)
    b = rng.standard_normal((batch, K, N), dtype=np.float32) * np.float32(0.1)
    x = be.transpose(be.from_numpy(np.ascontiguousarray(a.transpose(0, 2, 1))), 1, 2) if a_rows_fast else be.from_numpy(a)
    y = be.from_numpy(b) if b_rows_fast else be.transpose(be.from_numpy(np.ascontiguousarray(b.transpose(0, 2, 1))), 1, 2)
    return a, b, x, y


def check(got, a, b):
    a, b = a.astype(np.float64), b.astype(np.float64)
    K = a.shape[-1]
    # three left-out products of pieces (2^-24 together at most), a rounding per 16 values of k and kept product, and up to 16
    # partial sums, each relative to the sum of magnitudes
    bound = (1.0 + 6 * ((K + 15) // 16) + 16) * 2.0 ** -24 * (np.abs(a) @ np.abs(b)) + 1e-37
    assert (np.abs(got - a @ b) <= bound).all()


@pytest.mark.parametrize("size", SIZES, ids=str)
@pytest.mark.parametrize("layout", ["nt", "nn", "tt", "tn"])
def test_layouts_and_edges(hip, size, layout):
    M, K, N = size
    a, b, x, y = operands(hip, M, K, N, layout[0] == "t", layout[1] == "n")
    check(hip.to_numpy(hip.matmul(x, y)), a, b)


def test_batches_and_unaligned_views(hip):
    a, b, x, y = operands(hip, 70, 200, 90, False, False, batch=3)
    check(hip.to_numpy(hip.matmul(x, y)), a, b)
    x, y = hip.slice(x, 2, 3, 190), hip.slice(y, 1, 3, 190)   # rows begin 12 bytes behind a multiple of 16
    check(hip.to_numpy(hip.matmul(x, y)), a[:, :, 3:193], b[:, 3:193])


def test_a_row_of_the_unit_matrix_hands_values_through(hip):
    rng = np.random.default_rng(5)
    w = rng.standard_normal((1, 96, 200), dtype=np.float32) * np.exp(rng.uniform(-20, 20, (1, 96, 200))).astype(np.float32)
    eye = np.eye(96, dtype=np.float32)[None]
    np.testing.assert_array_equal(hip.to_numpy(hip.matmul(hip.from_numpy(eye), hip.from_numpy(w))), w)


@pytest.mark.parametrize("M", [16, 40, 130])
@pytest.mark.parametrize("side", ["left", "right"])
def test_ends_of_the_range(hip, M, side):
    """Infinities, values that round up beyond bfloat16's largest, rows of tiny values, NaN: as in 32-bit arithmetic."""
    K, N = 64, 130
    rng = np.random.default_rng(M)
    a = rng.standard_normal((1, M, K), dtype=np.float32)
    b = np.zeros((1, K, N), dtype=np.float32)
    b[0, rng.integers(0, K, N), np.arange(N)] = rng.choice(np.float32([1.0, -0.5, 2.0 ** -10]), N)   # a scaled choice: exact products
    a[0, 3] = np.float32(3.4028235e38) * np.sign(a[0, 3])
    a[0, 5] *= np.float32(1e-34)
    a[0, 7, 1] = np.inf
    a[0, 9, 2] = np.nan
    with np.errstate(invalid="ignore", over="ignore"):
        want = (a[0].astype(np.float64)[:, :, None] * b[0].astype(np.float64)[None]).sum(1).astype(np.float32)
    if side == "left":
        got = hip.to_numpy(hip.matmul(hip.from_numpy(a), hip.from_numpy(b)))[0]
    else:
        got = hip.to_numpy(hip.matmul(hip.transpose(hip.from_numpy(np.ascontiguousarray(b.transpose(0, 2, 1)).reshape(1, N, K)), 1, 1),
                                      hip.transpose(hip.from_numpy(a), 1, 2)))[0].T
    assert np.array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(got[~np.isnan(want)], want[~np.isnan(want)])


# the 128 x 128 tile; 64 x 64 of four waves (nt) and of two; 32 x 256 and 128 x 128 cut along k; 64 x 64 cut; 64 x 64 for any alignment;
# 256 x 256; 64 x 128 and 128 x 128; 128 x 128 for any alignment
TILES = [(2048, 64, 8192), (72, 64, 2048), (32, 64, 8192), (32, 2048, 8192), (200, 512, 256), (130, 63, 130), (2048, 128, 8192), (1024, 64, 4096), (1030, 63, 4098)]


def check_chosen(be, size, layout, rows, scales):
    """Every column of the right operand holds one value (a power of two): every result is one product, exact or out of range."""
    M, K, N = size
    rng = np.random.default_rng(M + K + N)
    a, b = rng.standard_normal((M, K), dtype=np.float32), np.zeros((K, N), dtype=np.float32)
    at, s = rng.integers(0, K, N), rng.choice(np.float32(scales), N)
    b[at, np.arange(N)] = s
    for r, make in rows.items():
        a[r] = make(rng, K)
    with np.errstate(all="ignore"):
        want = a[:, at].astype(np.float64) * s
        want = want.astype(np.float32)
        others = np.isfinite(a).sum(1)[:, None] - np.isfinite(a[:, at]) < K - 1   # infinity (or NaN) times zero among the terms
        want[others] = np.nan
    x = be.transpose(be.from_numpy(np.ascontiguousarray(a.T)), 0, 1) if layout[0] == "t" else be.from_numpy(a)
    y = be.from_numpy(b) if layout[1] == "n" else be.transpose(be.from_numpy(np.ascontiguousarray(b.T)), 0, 1)
    got = be.to_numpy(be.matmul(x, y))
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(got[~np.isnan(want)], want[~np.isnan(want)])


def one(value):
    def make(rng, K):
        r = rng.standard_normal(K, dtype=np.float32)
        r[K // 3] = value
        return r
    return make


@pytest.mark.parametrize("size", TILES, ids=str)
@pytest.mark.parametrize("layout", ["nt", "nn", "tt", "tn"])
def test_rows_at_the_ends_of_the_range(hip, size, layout):
    last = size[0] - 1
    check_chosen(hip, size, layout, {
        last: lambda rng, K: np.float32(3.4028235e38) * rng.choice(np.float32([1, -1]), K), 5: lambda rng, K: rng.standard_normal(K, dtype=np.float32) * np.float32(1e-34),
        last // 2: one(np.inf), last // 3: one(np.nan), last - 3: one(-np.inf)}, [1.0, -0.5, 2.0 ** -10])


@pytest.mark.parametrize("size", TILES, ids=str)
@pytest.mark.parametrize("layout", ["nt", "nn", "tt", "tn"])
def test_products_beyond_the_range(hip, size, layout):
    """Finite values whose products are infinite have the product's sign, whatever the pieces' are."""
    last = size[0] - 1
    signs = lambda rng, K: np.float32(1.01e22) * rng.choice(np.float32([1, -1]), K)    # noqa: E731  (a second piece of the other sign)
    check_chosen(hip, size, layout, {last: signs, 3: signs, last // 2: one(-1.1e38)}, [1.0, 2.0 ** 70, -2.0 ** 70])


@pytest.mark.parametrize("size,layout", [((512, 576, 1536), "nt"), ((512, 576, 1536), "nn"), ((512, 576, 1536), "tt"), ((512, 576, 1536), "tn"), ((1024, 1024, 2048), "nt"),
                                         ((4096, 256, 4096), "nt"), ((4096, 256, 4096), "tn"), ((1023, 2047, 513), "nt"), ((30, 1024, 8192), "nt")], ids=str)
def test_roundings_have_no_direction(hip, size, layout):
    """The error's mean over all results, against their root mean square: a rounding to nearest per 16 values of k has none (over
    these numbers of results its mean is below 2^-28), sums cut off below have 2^-27 and more."""
    a, b, x, y = operands(hip, *size, layout[0] == "t", layout[1] == "n", seed=3)
    want = a.astype(np.float64) @ b.astype(np.float64)
    d = hip.to_numpy(hip.matmul(x, y)) - want
    assert abs(d.mean()) <= 2.0 ** -28 * np.sqrt((want ** 2).mean()), d.mean() / np.sqrt((want ** 2).mean())


@pytest.mark.parametrize("size", TILES, ids=str)
@pytest.mark.parametrize("layout", ["nt", "nn", "tt", "tn"])
def test_small_values_beside_large_ones(hip, size, layout):
    """All bits of values down to the smallest subnormal, in rows that also hold ordinary ones."""
    def mixed(low, high):
        def make(rng, K):
            r = rng.standard_normal(K, dtype=np.float32)
            small = rng.random(K) < 0.7
            return np.where(small, np.ldexp(1 + rng.random(K), rng.integers(low, high, K)) * rng.choice([1, -1], K), r).astype(np.float32)
        return make

    last = size[0] - 1
    check_chosen(hip, size, layout, {last: mixed(-126, -100), 3: mixed(-149, -126), last // 2: mixed(-120, -110), last // 3: mixed(-149, 20)},
                 [1.0, -0.5, 2.0 ** 60, -2.0 ** -7])


def test_sums_of_small_and_large_products(hip):
    rng = np.random.default_rng(9)
    M, K, N = 150, 96, 200
    a = np.ldexp(rng.standard_normal((1, M, K)), rng.integers(-126, -120, (1, M, K))).astype(np.float32)
    b = np.ldexp(rng.standard_normal((1, K, N)), rng.integers(95, 100, (1, K, N))).astype(np.float32)
    a[0, :, 0], b[0, 0] = 1.0, 0.0          # a row's largest value meets nothing
    check(hip.to_numpy(hip.matmul(hip.from_numpy(a), hip.from_numpy(b))), a, b)
