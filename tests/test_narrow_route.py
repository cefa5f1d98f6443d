"""Which kernels a product of a narrow dtype is sent to: an operand that is not to be read as 32-bit words is on a kernel that reads
patterns, and that kernel reaches all of it.  The decision alone (a header without device code), so that matrices of 4 GiB need no memory."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "catgrad_amd", "csrc")
WORDS, LOW, WIDE = 0, 1, 2
BF16, F16, F8 = 1, 2, 3


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    d = tmp_path_factory.mktemp("route")
    (d / "route.cpp").write_text('''
#include "narrow_route.hpp"
extern "C" int route(int kind, int64_t m, int64_t x_pitch, int x_lies, int64_t n, int64_t y_pitch, int y_lies, int64_t k, int big, int wide_only) {
    return (int)cg::narrow_route(kind, {m, x_pitch, x_lies != 0}, {n, y_pitch, y_lies != 0}, k, true, big != 0, wide_only != 0);
}
extern "C" int64_t wide(int64_t units, int kind, int64_t m, int64_t n) { return cg::wide_columns(units, kind, m, n); }
extern "C" int fits(int kind, int64_t xp, int64_t m, int64_t wp, int64_t n, int64_t k) { return cg::fits_narrow_tiles(kind, xp, m, wp, n, k); }
''')
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, "-o", str(d / "route.so"), str(d / "route.cpp")])
    lib = ctypes.CDLL(str(d / "route.so"))
    lib.route.argtypes = [ctypes.c_int, *[ctypes.c_int64] * 2, ctypes.c_int, *[ctypes.c_int64] * 2, ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_int]
    lib.wide.argtypes, lib.wide.restype = [ctypes.c_int64, ctypes.c_int, *[ctypes.c_int64] * 2], ctypes.c_int64
    lib.fits.argtypes = [ctypes.c_int, *[ctypes.c_int64] * 5]
    return lib


@pytest.mark.parametrize("kind,m,n,k,x_lies,y_lies,want", [
    (BF16, 64, 512, 2048, 0, 1, LOW),                 # activations in words, weights as they lie
    (F16, 300, 260, 64, 1, 0, LOW),
    (BF16, 64, 512, 2048, 0, 0, WORDS),               # nothing lies narrow
    (BF16, 64, 262144, 8192, 0, 1, WORDS),            # weights of exactly 4 GiB
    (BF16, 64, 262143, 8192, 0, 1, LOW),              # a row less
    (BF16, 64, 262144, 8192, 1, 0, WORDS),            # the same matrix, packed for the product
    (BF16, 1 << 20, 200, 2048, 1, 1, WORDS),          # activations of 4 GiB
    (F8, 64, 524288, 8192, 0, 1, WORDS),
    (F8, 64, 524287, 8192, 0, 1, LOW),
    (BF16, 64, 1 << 30, 1 << 33, 0, 1, WORDS),        # beyond what an index holds
])
def test_narrow_operands_stay_within_reach(route, kind, m, n, k, x_lies, y_lies, want):
    assert route.route(kind, m, k, x_lies, n, k, y_lies, k, 0, 0) == want
    assert route.route(kind, m, k, x_lies, n, k, y_lies, k, 0, 1) == WORDS    # asked for the wide tiles alone
    assert route.route(kind, m, k, x_lies, n, k, y_lies, k, 1, 0) == WIDE


def test_pitches(route):
    assert route.route(BF16, 64, 2048, 1, 512, 4096, 1, 2048, 0, 0) == LOW                 # rows of a wider matrix
    assert route.route(BF16, 64, 2048, 1, 1 << 16, 1 << 15, 1, 2048, 0, 0) == WORDS        # whose rows span 4 GiB
    assert route.route(BF16, 64, 2052, 1, 512, 2048, 1, 2048, 0, 0) == WORDS               # rows off 16 bytes
    assert route.route(BF16, 64, 2052, 0, 512, 2048, 1, 2048, 0, 0) == LOW                 # (packed: its own pitch does not count)
    for kind, k in ((BF16, 2044), (F8, 2056), (BF16, 0)):
        assert not route.fits(kind, k, 64, k, 512, k)


def test_columns_left_to_the_narrow_tiles(route):
    """At most five sixteenths of a round of 256-wide tiles move, and what stays is no round that is nearly empty either."""
    moved = set()
    for units in (256, 304):
        for m in (256, 300, 1024, 1030, 2048, 5000, 7424, 8192, 16384, 33000, 66600, 1 << 20):
            for n in (200, 256, 500, 700, 1000, 1300, 2052, 2816, 4000, 8256, 10240, 12288, 16484, 20480, 24576, 65600, 131000):
                assert route.wide(units, F8, m, n) == n
                kept, rows, tiles = route.wide(units, BF16, m, n), -(-m // 256), -(-m // 256) * -(-n // 256)
                if kept == n:
                    continue
                assert 0 < kept < n and kept % 256 == 0
                if units == 256:
                    moved.add((m, n))
                stays = rows * kept // 256
                assert (tiles - stays) * 16 <= 5 * units and (stays % units == 0 or stays % units * 16 >= 11 * units)
    assert {(1024, 16484), (2048, 8256), (2048, 10240), (8192, 2052), (300, 65600), (5000, 4000)} <= moved
    assert not {(66600, 500), (7424, 2816), (1024, 24576), (2048, 12288)} & moved
