"""Attention or a row sum whose launch waits for the next call holds memory meanwhile: a call that finds no room takes that memory first, as it would
have been there had nothing waited.  A second process, in which the library's device memory is limited to a total."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
#include <map>
#include <mutex>
static std::mutex mu;
static std::map<void *, size_t> sizes;
static size_t used = 0, most = ~(size_t)0;
static int refused = 0;
static void *next(const char *name) {
    void *runtime = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
    return runtime ? dlsym(runtime, name) : nullptr;
}
extern "C" {
void room(long n) { most = n < 0 ? ~(size_t)0 : used + n, refused = 0; } // from now on so many bytes more than there are
int count(void) { return refused; }
int hipMalloc(void **p, size_t n) {
    static const auto to = (int (*)(void **, size_t))next("hipMalloc");
    std::lock_guard<std::mutex> lk(mu);
    if (used + n > most) return refused++, *p = nullptr, 2;     /* out of memory */
    const int rc = to ? to(p, n) : 999;
    if (!rc) sizes[*p] = n, used += n;
    return rc;
}
int hipFree(void *p) {
    static const auto to = (int (*)(void *))next("hipFree");
    {
        std::lock_guard<std::mutex> lk(mu);
        const auto at = sizes.find(p);
        if (at != sizes.end()) used -= at->second, sizes.erase(at);
    }
    return to ? to(p) : 999;
}
}
"""

PROGRAM = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)        # before the library: its requests come here first
shim.room.argtypes = [ctypes.c_long]
sys.path.insert(0, sys.argv[2])
import numpy as np
import block_cases as C
from catgrad_amd import HipBackend
be = HipBackend(0)


def step(room):
    '''Attention of a token, then experts.  Its segments' results are 6 MB, what the experts need a few hundred KB.'''
    rng = np.random.default_rng(0)
    heads, kv_heads, dim, width, ff, cached = 16, 8, 128, 256, 16384, 6000
    o = C.turned(heads, kv_heads, dim, dim, 16)
    t = C.attention_case(rng, 1, 2, o, norms=False)
    caches = [be.from_numpy(rng.standard_normal((1, kv_heads, cached, dim)).astype(np.float32)) for _ in range(2)]
    e = C.expert_case(rng, 1, width, 4, ff, "f32")
    ex = {n: be.from_numpy(e[n].reshape((1, 1, -1) if n == "logits" else e[n].shape)) for n in ("logits", "correction", "gate_up", "down")}
    ex["h"] = be.from_numpy(e["h"].reshape(1, 1, width))
    w, x = be.from_numpy((rng.standard_normal((width, heads * dim)) * 0.02).astype(np.float32)), be.from_numpy(rng.standard_normal((1, 1, width)).astype(np.float32))
    parts = [{n: be.from_numpy(t[n][:, s:s + 1] if n != "talk" else t[n]) for n in ("q", "k", "v", "talk")} for s in range(2)]
    y, k, v = be.block_attention({**parts[0], "k_cache": caches[0].move(), "v_cache": caches[1].move()}, position=cached, **o)  # (makes room for more keys)
    del y
    for a in list(ex.values()) + [w, x] + list(parts[1].values()):
        be.realize(a)
    be.pool_trim()
    y, k, v = be.block_attention({**parts[1], "k_cache": k.move(), "v_cache": v.move()}, position=cached + 1, **o)
    shim.room(room)
    out = be.block_residual(x, [{"y": y.move(), "w": w}], scale=0.4, experts=ex, top=2, groups=1, keep=1, limit=1.2, slope=1.702)
    seen = shim.count()
    shim.room(-1)
    return [be.to_numpy(a) for a in (out, k, v)], seen


def row_sum(room):
    '''The sum behind the tokens' own vectors, then filters.  Its second term is 128 KB, as is what the filters leave for their product.'''
    rng = np.random.default_rng(1)
    B, W, dim, taps = 8, 4096, 64, 4
    f = lambda *s: be.from_numpy(rng.standard_normal(s).astype(np.float32))
    side = {"x": f(B, 1, W), "ids": be.from_numpy(rng.integers(0, 9, (B, 1), dtype=np.uint32)), "table": f(9, dim), "gate": f(dim, W), "proj": f(W, dim), "norm": f(W)}
    state, one = f(B, taps - 1, W), {"gamma": f(W), "conv": f(W, taps), "w": f(8, W)}
    for a in list(side.values()) + [state] + list(one.values()):
        be.realize(a)
    be.pool_trim()
    z = be.block_token_side(side, first=0, eps=2e-3, scale=0.02)
    shim.room(room)
    y, h, s = be.block_conv_linear(z, state, [{**one, "keep": 0}], groups=4, eps=2e-3)
    seen = shim.count()
    shim.room(-1)
    return [be.to_numpy(a) for a in [z, s] + y], seen


for f, room in ((step, 0), (row_sum, (3 * 8 * 4096 * 4) + (16 << 10))):
    want, seen = f(-1)
    assert not seen
    got, seen = f(room)
    print(f.__name__, "requests refused:", seen, flush=True)
    assert seen
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
print("done", flush=True)
"""


def test_no_room_but_what_waits(tmp_path):
    here = os.path.dirname(os.path.abspath(__file__))
    (tmp_path / "shim.cpp").write_text(SHIM)
    (tmp_path / "program.py").write_text(PROGRAM)
    subprocess.check_call(["g++", "-shared", "-fPIC", "-o", str(tmp_path / "shim.so"), str(tmp_path / "shim.cpp"), "-ldl"])
    env = dict(os.environ, PYTHONPATH=os.path.dirname(here))
    r = subprocess.run([sys.executable, str(tmp_path / "program.py"), str(tmp_path / "shim.so"), here], env=env, capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0 and r.stdout.endswith("done\n")
