"""Launches that are refused behind the call that asked for them: the next wait says which one and why, once, and nothing of it is a later call's;
what the host can tell before a launch is the call's own error.  A second process, in which chosen requests to the runtime are refused
(no kernel runs that should not)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
#include <atomic>
struct dim { unsigned x, y, z; };
static std::atomic<int> launch{0}, attribute{0}, refused{0};
static void *next(const char *name) {
    void *runtime = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
    return runtime ? dlsym(runtime, name) : nullptr;
}
extern "C" {
void refuse_launch(int code) { refused = 0, launch = code; }        // the next launch comes to `code`
void refuse_attribute(int code) { refused = 0, attribute = code; }  // so does every reservation, until it is 0 again
int count(void) { return refused; }
int hipLaunchKernel(const void *f, dim g, dim b, void **a, size_t l, void *s) {
    if (const int code = launch.exchange(0)) return refused++, code;
    static const auto to = (int (*)(const void *, dim, dim, void **, size_t, void *))next("hipLaunchKernel");
    return to ? to(f, g, b, a, l, s) : 999;
}
int hipFuncSetAttribute(const void *f, int what, int value) {
    if (attribute) return refused++, attribute.load();
    static const auto to = (int (*)(const void *, int, int))next("hipFuncSetAttribute");
    return to ? to(f, what, value) : 999;
}
}
"""

PROGRAM = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)        # before the library: its requests come here first
sys.path.insert(0, sys.argv[2])
import numpy as np
import block_cases as C
from catgrad_amd import BackendPanic, HipBackend
be = HipBackend(0)


def error(f, *a):
    try:
        f(*a)
    except BackendPanic as e:
        return str(e)
    return None


def chain(n):
    y, w = be.from_numpy(np.ones((1, 12, 64), dtype=np.float32)), be.from_numpy(np.eye(64, dtype=np.float32)[None])
    for _ in range(n):
        y = be.matmul(y, w)
    return y


def refused(wait, before=lambda: None):
    be.sync()
    y = chain(40)                     # from here on launches are the thread's
    kept = before()
    shim.refuse_launch(9)
    y = chain(40)
    got = error(wait, y)
    assert shim.count() == 1, shim.count()
    assert got and "HIP error 9" in got and "_kernel" in got, got
    assert error(be.sync) is None     # reported once, and with it whatever the kernels had found
    z = chain(3)
    assert np.array_equal(be.to_numpy(z), np.ones((1, 12, 64), dtype=np.float32))


refused(lambda y: be.sync())
refused(be.to_numpy)
print("launches", flush=True)
table, far = be.from_numpy(np.zeros((5, 8), dtype=np.float32)), be.from_numpy(np.array([9], dtype=np.uint32))
refused(lambda y: be.sync(), lambda: be.realize(be.index(table, 0, far)))
refused(be.to_numpy, lambda: be.realize(be.index(table, 0, far)))
be.realize(be.index(table, 0, far))
assert "out of bounds" in error(be.sync)
print("with a fault", flush=True)

# attention over mixed scores whose launch waits for the next call: 71 KB of LDS to be reserved
o = C.turned(32, 16, 128, 64, 16)
t = C.attention_case(np.random.default_rng(0), 1, 6, o, norms=False)
def attention():
    c = {n: be.from_numpy(np.ones((1, 16, 5, d), dtype=np.float32)) for n, d in (("k_cache", 128), ("v_cache", 64))}
    y, k, v = be.block_attention({**{n: be.from_numpy(t[n]) for n in ("q", "k", "v", "talk")}, **c}, position=5, **o)
    return y
shim.refuse_attribute(9)
got = error(attention)
assert shim.count() > 0
shim.refuse_attribute(0)
assert got and "HIP error 9" in got, got
assert error(be.sync) is None
assert np.isfinite(be.to_numpy(attention())).all()
print("done", flush=True)
"""


def test_refused(tmp_path):
    here = os.path.dirname(os.path.abspath(__file__))
    (tmp_path / "shim.cpp").write_text(SHIM)
    (tmp_path / "program.py").write_text(PROGRAM)
    subprocess.check_call(["g++", "-shared", "-fPIC", "-o", str(tmp_path / "shim.so"), str(tmp_path / "shim.cpp"), "-ldl"])
    env = dict(os.environ, PYTHONPATH=os.path.dirname(here))
    r = subprocess.run([sys.executable, str(tmp_path / "program.py"), str(tmp_path / "shim.so"), here], env=env, capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0 and r.stdout.endswith("done\n")
