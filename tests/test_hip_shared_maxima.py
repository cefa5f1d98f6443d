"""Row maxima that are subtracted from their rows and read again (log-sum-exp op by op): taken in the program's kernel while the row is
in its registers.  Against float64, with the maxima moved, kept and read, and with every other consumer of their broadcast."""
import numpy as np
import pytest

from catgrad_amd import _abi as A

pytestmark = pytest.mark.gpu

# rows beside columns: one item a lane, odd counts, the edges of what a lane keeps in registers (12 x 256, 8192, 16384 values), longer
# rows, a few long ones
SHAPES = [(1, 16), (3, 127), (927, 235), (5, 512), (7, 3072), (6, 3076), (9, 8192), (130, 8196), (70, 16384), (66, 16388), (65, 40000), (2, 40000), (3, 8191)]


def _x(rows, cols, special):
    rng = np.random.default_rng(rows * 7 + cols)
    x = (rng.standard_normal((rows, cols)) * 3).astype(np.float32)
    if special:
        x[0, ::3] = -np.inf
        if rows > 1:
            x[1] = -np.inf
        if rows > 2:
            x[2, cols // 2] = np.inf
        if rows > 3:
            x[3, cols - 1] = np.nan
        if rows > 4:
            x[4] = 80.0
    return x


def _want(x):
    w = x.astype(np.float64)
    # the program's own order: maxima start from the lowest finite value and pass over NaN
    m = np.maximum(np.fmax.reduce(w, -1, keepdims=True), np.float64(np.finfo(np.float32).min))
    with np.errstate(all="ignore"):
        d = w - m
        e = np.exp(d)
        return m, d, e, np.log(e.sum(-1, keepdims=True)) + m


def _close(got, want, n):
    # exp, log and the last addition by a few 2^-24 of their results, the sum by its longest chain (a lane's values, the lanes)
    tol = (n / 256 + 32) * 2.0 ** -24
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    ok = np.isfinite(want)
    np.testing.assert_array_equal(got[~ok & ~np.isnan(want)], want[~ok & ~np.isnan(want)].astype(np.float32))
    assert (np.abs(got[ok] - want[ok]) <= tol * np.maximum(np.abs(want[ok]), 1.0)).all()


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_log_sum_exp_and_what_is_left_of_it(hip, rows, cols, special):
    x = _x(rows, cols, special)
    m, d, e, lse = _want(x)
    n, shape = cols, (rows, cols)

    def shifted(t, mx):
        return hip.sub(t, hip.broadcast(mx, shape).move())

    tx = hip.from_numpy(x)
    mx = hip.max(tx)                                                    # moved in the end: no launch of its own
    out = hip.log(hip.sum(hip.exp(shifted(tx, mx).move()).move()).move())
    _close(hip.to_numpy(hip.add(out.move(), mx.move())), lse, n)
    mx = hip.max(tx)                                                    # kept, and read afterwards
    out = hip.add(hip.log(hip.sum(hip.exp(shifted(tx, mx).move()).move()).move()).move(), mx)
    _close(hip.to_numpy(out), lse, n)
    np.testing.assert_array_equal(hip.to_numpy(mx), m.astype(np.float32))
    mx = hip.max(tx)                                                    # read in between
    sh = shifted(tx, mx)
    np.testing.assert_array_equal(hip.to_numpy(mx), m.astype(np.float32))
    _close(hip.to_numpy(sh), d, n)
    mx = hip.max(tx)
    _close(hip.to_numpy(hip.exp(shifted(tx, mx).move())), e, n)
    _close(hip.to_numpy(mx), m, n)


@pytest.mark.parametrize("rows,cols", [(5, 512), (9, 8192), (3, 127)])
def test_other_consumers_of_the_broadcast(hip, rows, cols):
    x, y = _x(rows, cols, False), _x(rows, cols, False)[::-1].copy()
    m = x.max(-1, keepdims=True)
    shape = (rows, cols)
    tx, ty = hip.from_numpy(x), hip.from_numpy(y)
    mx = hip.max(tx)
    np.testing.assert_array_equal(hip.to_numpy(hip.broadcast(mx, shape)), np.broadcast_to(m, shape))
    mx = hip.max(tx)
    np.testing.assert_array_equal(hip.to_numpy(hip.sub(ty, hip.broadcast(mx, shape).move())), y - m)   # another left side
    mx = hip.max(tx)
    np.testing.assert_array_equal(hip.to_numpy(hip.sub(hip.broadcast(mx, shape).move(), tx)), m - x)   # the other way round
    mx = hip.max(tx)
    b = hip.broadcast(mx, shape)                                                                      # a broadcast that is held
    np.testing.assert_array_equal(hip.to_numpy(hip.sub(tx, b)), x - m)
    np.testing.assert_array_equal(hip.to_numpy(hip.mul(tx, b)), x * m)
    np.testing.assert_array_equal(hip.to_numpy(hip.transpose(b, 0, 1)), np.broadcast_to(m, shape).T)
    np.testing.assert_array_equal(hip.to_numpy(hip.max(hip.transpose(b, 0, 1).move()))[:, 0], np.full(cols, m.max()))
    mx = hip.max(tx)
    b = hip.broadcast(mx, shape)
    np.testing.assert_array_equal(hip.to_numpy(hip.max(b)), m)
    mx = hip.max(tx)
    b = hip.concat(hip.broadcast(mx, shape).move(), ty, 1)
    np.testing.assert_array_equal(hip.to_numpy(b), np.concatenate([np.broadcast_to(m, shape), y], 1))
    t = hip.transpose(tx, 0, 1)                                                                       # rows that do not lie in a row
    mt = hip.max(t)
    got = hip.sub(t, hip.broadcast(mt, (cols, rows)).move())
    np.testing.assert_array_equal(hip.to_numpy(got), x.T - x.T.max(-1, keepdims=True))


@pytest.mark.parametrize("rows,cols", [(70, 8192), (9, 130), (5, 64), (200, 24), (1, 33)])
def test_programs_around_shared_maxima(hip, rows, cols):
    """Every way on from x - max x: right, and the maxima taken anew only in a program that is compiled; the interpreter reads them,
    from the reduction's own kernel (a launch of that class)."""
    x, z = _x(rows, cols, False), _x(rows, cols, False)[:, ::-1].copy()
    x[0, 0] = 9.0
    m, d, e, lse = _want(x)
    tx, tz, shape = hip.from_numpy(x), hip.from_numpy(z), (rows, cols)
    half = hip.broadcast(hip.ndarray_from_vec_f32([0.5], ()), shape)
    total = e.sum(-1, keepdims=True)
    ways = {  # name: (what is made of x - max x and the maxima, its value, whether its program is a compiled one)
        "shift": (lambda s, mx: s, d, True),
        "exp": (lambda s, mx: hip.exp(s.move()), e, True),
        "scaled": (lambda s, mx: hip.mul(s.move(), half), d * 0.5, False),
        "temperature": (lambda s, mx: hip.exp(hip.mul(s.move(), half).move()), np.exp(d * 0.5), False),
        "of_another": (lambda s, mx: hip.mul(s.move(), tz), d * z, False),
        "sum": (lambda s, mx: hip.sum(s.move()), d.sum(-1, keepdims=True), False),
        "largest": (lambda s, mx: hip.max(s.move()), np.zeros_like(m), False),
        "sum_of_exp": (lambda s, mx: hip.sum(hip.exp(s.move()).move()), total, False),
        "log_sum": (lambda s, mx: hip.log(hip.sum(hip.exp(s.move()).move()).move()), np.log(total), False),
        "log_sum_exp_twice": (lambda s, mx: hip.mul(hip.add(hip.log(hip.sum(hip.exp(s.move()).move()).move()).move(), mx).move(),
                                                    hip.broadcast(hip.ndarray_from_vec_f32([2.0], ()), (rows, 1)).move()), 2 * lse, False),
        "maxima_first": (lambda s, mx: hip.add(mx, hip.log(hip.sum(hip.exp(s.move()).move()).move()).move()), lse, False),
        "minus_log_sum": (lambda s, mx: hip.sub(s, hip.broadcast(hip.log(hip.sum(hip.exp(s).move()).move()).move(), shape).move()), d - np.log(total), None),
        "soft_max": (lambda s, mx: (lambda ex: hip.div(ex, hip.broadcast(hip.sum(ex), shape).move()))(hip.exp(s.move())), e / total, None),
        "maxima_again": (lambda s, mx: hip.sub(s.move(), hip.broadcast(mx, shape).move()), d - m, False),
        "turned": (lambda s, mx: hip.exp(hip.transpose(s.move(), 0, 1).move()), e.T, False),
        "part": (lambda s, mx: hip.exp(hip.slice(s.move(), 1, 1, cols - 3).move()), e[:, 1:cols - 2], False),
        "reshaped": (lambda s, mx: hip.exp(hip.reshape(s.move(), (rows * cols, 1)).move()), e.reshape(-1, 1), False),
        "beside": (lambda s, mx: hip.concat(s.move(), tz, 1), np.concatenate([d, z], 1), False),
        "above": (lambda s, mx: hip.concat(tz, s.move(), 0), np.concatenate([z, d], 0), False),
        "rounded": (lambda s, mx: hip.cast(s.move(), A.BF16), d, False),
        "held": (lambda s, mx: hip.add(s, hip.exp(s).move()), d + e, None),
        "where": (lambda s, mx: hip.where_cond(hip.lt(s, tz).move(), s, tz), np.minimum(d.astype(np.float32), z), None),
    }
    hip.profile_enable(A.K_REDUCE)
    try:
        for name, (way, want, compiled) in ways.items():
            for kept in (True, False):
                mx = hip.max(tx)
                s = hip.sub(tx, hip.broadcast(mx, shape).move())
                hip.sync()
                hip.profile_read(A.K_REDUCE)
                y = way(s, mx)
                if not kept:
                    del mx, s
                hip.realize(y)
                hip.sync()
                launches = hip.profile_read(A.K_REDUCE)[0]
                if compiled is not None and cols > 32:
                    assert (launches == 0) == compiled, (name, kept, launches)
                got = hip.to_numpy(hip.cast(y, A.F32))
                if name == "rounded":
                    assert (np.abs(got - want) <= 2.0 ** -8 * np.abs(want)).all(), name
                else:
                    tol = (cols / 256 + 32) * 2.0 ** -23
                    assert (np.abs(got - want) <= tol * np.maximum(np.abs(want), np.abs(x).max() + np.abs(z).max())).all(), name
                if kept:
                    np.testing.assert_array_equal(hip.to_numpy(mx), m.astype(np.float32))
    finally:
        hip.profile_enable(A.K_REDUCE, 0)


@pytest.mark.parametrize("rows,cols", [(300, 4096), (70, 16384), (9, 130)])
def test_rows_that_lie_in_two_bytes(hip, rows, cols):
    x = _x(rows, cols, False)
    bits = (x.view(np.uint32) >> 16).astype(np.uint16)
    x = (bits.astype(np.uint32) << 16).view(np.float32)
    tx = hip.cast(hip.ndarray_from_vec_bf16(bits, (rows, cols)).move(), A.F32)
    mx = hip.max(tx)
    e = hip.exp(hip.sub(tx, hip.broadcast(mx, (rows, cols)).move()).move())
    got = hip.to_numpy(hip.add(hip.log(hip.sum(e.move()).move()).move(), mx.move()))
    _close(got, _want(x)[3], cols)


@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 1100, 4097, 16383, 16384, 16385])
def test_small_read_backs(hip, n):
    x = np.random.default_rng(n).standard_normal(n + 3).astype(np.float32)
    t = hip.from_numpy(x)
    np.testing.assert_array_equal(hip.to_numpy(hip.slice(t, 0, 0, n)), x[:n])
    np.testing.assert_array_equal(hip.to_numpy(hip.slice(t, 0, 3, n)), x[3:])     # from an address that is not a multiple of 16
