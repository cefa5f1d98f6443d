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
extern "C" int fits(int kind, int64_t xp, int64_t m, int64_t wp, int64_t n, int64_t k) { return cg::fits_narrow_tiles(kind, xp, m, wp, n, k); }
''')
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, "-o", str(d / "route.so"), str(d / "route.cpp")])
    lib = ctypes.CDLL(str(d / "route.so"))
    lib.route.argtypes = [ctypes.c_int, *[ctypes.c_int64] * 2, ctypes.c_int, *[ctypes.c_int64] * 2, ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_int]
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
