"""Calls whose scratch memory cannot be had give the results that they give with it: operands that are not packed are read as they
are, sums over k are not cut, caches are copied without a store behind them.  A second process, in which the library's requests for device memory of chosen sizes are refused."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
typedef int (*request)(void **, size_t);
static size_t from = 1, to = 0;
static int refused = 0;
void refuse(size_t a, size_t b) { from = a, to = b, refused = 0; }
int count(void) { return refused; }
int hipMalloc(void **p, size_t n) {
    if (n >= from && n <= to) return refused++, *p = 0, 2;  /* out of memory */
    static request next;
    if (!next) {
        void *runtime = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
        if (!runtime) return 999;
        next = (request)dlsym(runtime, "hipMalloc");
    }
    return next(p, n);
}
"""

PROGRAM = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)        # before the library: its requests come here first
shim.refuse.argtypes = [ctypes.c_size_t] * 2
import numpy as np
from catgrad_amd import HipBackend, _abi as A
be = HipBackend(0)
rng = np.random.default_rng(1)


def whole(*shape):
    return rng.integers(-3, 4, shape).astype(np.float32)        # sums that every order of summation gives alike


def upload(a, dtype):
    if dtype == A.F32:
        return be.from_numpy(a)
    if dtype == A.F16:
        return be.ndarray_from_vec_f16(a.astype(np.float16), a.shape)
    bits = a.view(np.uint32)
    if dtype == A.BF16:
        return be.ndarray_from_vec_bf16((bits >> 16).astype(np.uint16), a.shape)
    code = np.uint8([0, 0x38, 0x40, 0x44])                      # 0 .. 3 as E4M3
    return be.ndarray_from_vec_fp8(code[np.abs(a).astype(int)] | (bits >> 24 & 0x80).astype(np.uint8), a.shape)


# M, K, N, dtype, the sizes that are refused
for M, K, N, dtype, low, high in (
        (96, 512, 1024, A.BF16, 90_000, 140_000),               # 128-wide tiles, the left operand to be packed
        (96, 512, 1024, A.F16, 90_000, 140_000),
        (4096, 8, 2048, A.BF16, 20_000, 140_000),               # 256-wide tiles, both
        (96, 512, 1024, A.F8, 45_000, 60_000),
        (96, 4096, 1024, A.BF16, 700_000, 16 << 20),            # cut along k
        (32, 8192, 2048, A.F32, 400_000, 16 << 20)):
    a, b = whole(M, K), whole(N, K)
    x, w = upload(a[None], dtype), upload(b[None], dtype)
    y = be.transpose(w, 1, 2)
    want = be.from_numpy((a @ b.T)[None])
    want = be.to_numpy(be.cast(be.cast(want, dtype), A.F32) if dtype != A.F32 else want)
    be.pool_trim()
    shim.refuse(low, high)
    z = be.matmul(x, y)
    be.sync()
    seen = shim.count()
    shim.refuse(1, 0)
    assert np.array_equal(be.to_numpy(be.cast(z, A.F32)), want), (M, K, N, dtype)
    z = be.matmul(x, y)
    assert np.array_equal(be.to_numpy(be.cast(z, A.F32)), want), (M, K, N, dtype)
    print(M, K, N, dtype, "requests refused:", seen, flush=True)
    assert seen, (M, K, N, dtype)

# a cache, its dtype, the part of axis 2 that is appended to, the sizes that are refused, whether they are asked for at all
for shape, dtype, part, low, high, asked in (
        ((4, 4, 3, 256), A.F32, None, 500_000, 16 << 20, True),   # few tokens: a store with room for more
        ((4, 4, 80, 256), A.F32, None, 4 << 20, 64 << 20, True),  # many
        ((64, 16, 8, 128), A.BF16, 1, 3 << 20, 8 << 20, False)):  # a row of a tensor that lies in two bytes: not the words of all of it
    a = whole(*shape)
    row = whole(*shape[:2], 1, shape[3])
    x, y = upload(a, dtype), upload(row, dtype)
    if part is not None:
        x, a = be.slice(x, 2, part, 1), a[:, :, part:part + 1]
    be.pool_trim()
    shim.refuse(low, high)
    z = be.concat(x, y, 2)
    z = be.concat(z.move(), y, 2)
    be.sync()
    seen = shim.count()
    shim.refuse(1, 0)
    assert np.array_equal(be.to_numpy(be.cast(z, A.F32)), np.concatenate([a, row, row], 2)), shape
    print(shape, dtype, "requests refused:", seen, flush=True)
    assert bool(seen) == asked, shape

# sums and maxima of the rows of a tensor that lies in two bytes or one, as f32: neither its words nor a place for parts of rows is needed
for shape, dtype, turn, low, high, asked in (
        ((8, 262144), A.BF16, False, 10_000, 16 << 20, True),     # a few long rows: the parts
        ((8, 262140), A.F16, False, 4 << 20, 16 << 20, False),
        ((3, 400004), A.F8, False, 2 << 20, 16 << 20, False),
        ((40000, 64), A.BF16, True, 8 << 20, 16 << 20, False),    # rows that lie side by side
        ((1000, 2048), A.F8, True, 6 << 20, 16 << 20, False)):
    a = whole(*shape)
    x = upload(a, dtype)
    if turn:
        x, a = be.transpose(x, 0, 1), a.T
    for op, want in ((be.sum, a.sum(-1, keepdims=True)), (be.max, a.max(-1, keepdims=True))):
        be.pool_trim()
        shim.refuse(low, high)
        z = op(be.cast(x, A.F32).move())
        be.realize(z)
        be.sync()
        seen = shim.count()
        shim.refuse(1, 0)
        assert np.array_equal(be.to_numpy(z), want), shape
        print(shape, dtype, "requests refused:", seen, flush=True)
        assert bool(seen) == asked, shape
print("done", flush=True)
"""


def test_products_without_scratch_memory(tmp_path):
    (tmp_path / "shim.c").write_text(SHIM)
    (tmp_path / "program.py").write_text(PROGRAM)
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", str(tmp_path / "shim.so"), str(tmp_path / "shim.c"), "-ldl"])
    env = dict(os.environ, PYTHONPATH=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    r = subprocess.run([sys.executable, str(tmp_path / "program.py"), str(tmp_path / "shim.so")], env=env, capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0 and r.stdout.endswith("done\n")
