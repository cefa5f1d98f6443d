"""A backend's launches go through a thread of its own when there are many between two waits of the host: whatever else is put on the
stream, allocated or given back in between stays in order, on every backend and from every thread."""
import os
import subprocess
import sys
import threading
import time

import numpy as np
import pytest

import block_cases as C
from catgrad_amd import BackendPanic, HipBackend

pytestmark = pytest.mark.gpu


def rolled(be, n, size=64):
    """n products with a permutation: rows that have moved on by n places, exactly."""
    x = np.arange(size * 12, dtype=np.float32).reshape(1, 12, size)
    w = be.from_numpy(np.roll(np.eye(size, dtype=np.float32), 1, axis=1)[None])
    y = be.from_numpy(x)
    for _ in range(n):
        y = be.matmul(y, w)
    return y, np.roll(x, n, axis=2)


@pytest.mark.parametrize("n", [1, 11, 12, 13, 14, 63, 64, 65, 77, 400])
def test_in_order(n):
    be = HipBackend(0)
    for _ in range(3):
        y, want = rolled(be, n)
        np.testing.assert_array_equal(be.to_numpy(y), want)
    be.close()


def test_between_copies_and_memory_given_back():
    be = HipBackend(0)
    rng = np.random.default_rng(0)
    big = rng.standard_normal((700, 1000), dtype=np.float32)     # uploads and read-backs by the runtime's copies
    for i in range(20):
        y, want = rolled(be, 40)
        a = be.from_numpy(big + np.float32(i))
        z, want2 = rolled(be, 40)
        b = be.add(a, be.from_numpy(big))
        if i % 5 == 0:
            be.pool_trim()
        np.testing.assert_array_equal(be.to_numpy(y), want)
        np.testing.assert_array_equal(be.to_numpy(b), (big + np.float32(i)) + big)
        np.testing.assert_array_equal(be.to_numpy(z), want2)
    be.close()


def test_threads_and_backends():
    shared, wrong = HipBackend(0), []
    own = [HipBackend(0) for _ in range(3)]

    def work(be):
        for n in (5, 50, 100):
            y, want = rolled(be, n)
            wrong.extend([n] if not np.array_equal(be.to_numpy(y), want) else [])

    t = [threading.Thread(target=work, args=(shared if i % 2 else own[i // 2],)) for i in range(6)]
    for x in t:
        x.start()
    for x in t:
        x.join()
    assert not wrong
    for be in [shared] + own:
        be.close()


@pytest.mark.parametrize("held", [False, True])
@pytest.mark.parametrize("idle", [0, 0.005], ids=["awake", "asleep"])
def test_closed_with_launches_on_their_way(held, idle):
    """A backend that is closed finishes what was launched; tensors that outlive it are released behind it, the last one ends it."""
    for n in (5, 100):
        be = HipBackend(0)
        y, _ = rolled(be, n)
        if not held:
            del y
        time.sleep(idle)
        be.close()
        if held:
            with pytest.raises(BackendPanic):
                be.to_numpy(y)
            del y


def waiting_attention(be):
    o = C.turned(8, 4, 64, 64, 16)
    t = C.attention_case(np.random.default_rng(0), 1, 1, o, norms=False)
    caches = {n: be.from_numpy(np.ones((1, 4, 5, 64), dtype=np.float32)) for n in ("k_cache", "v_cache")}
    return be.block_attention({**{n: be.from_numpy(t[n]) for n in t}, **caches}, position=5, **o)


def waiting_sum(be):
    f = lambda *s: be.from_numpy(np.full(s, 0.5, dtype=np.float32))
    side = {"x": f(1, 1, 1024), "ids": be.from_numpy(np.zeros((1, 1), dtype=np.uint32)), "table": f(9, 64), "gate": f(64, 1024), "proj": f(1024, 64), "norm": f(1024)}
    return be.block_token_side(side, first=0, eps=2e-3, scale=0.02)


@pytest.mark.parametrize("held", [False, True])
@pytest.mark.parametrize("what", [waiting_attention, waiting_sum], ids=lambda f: f.__name__)
def test_closed_with_a_launch_that_waits(what, held):
    for _ in range(3):
        be = HipBackend(0)
        r = what(be)
        if not held:
            del r
        be.close()
        if held:
            del r


def test_process_ends_with_launches_on_their_way():
    code = ("import sys; sys.path[:0] = ['.', 'tests']\nimport numpy as np\nfrom test_hip_launch_thread import HipBackend, rolled, waiting_attention\n"
            "be = HipBackend(0); y, _ = rolled(be, 300); r = waiting_attention(be); print('end', flush=True)")
    for _ in range(3):
        r = subprocess.run([sys.executable, "-c", code], cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))), capture_output=True, text=True, timeout=100)
        assert r.returncode == 0 and r.stdout == "end\n", (r.returncode, r.stderr)


def test_without_the_thread():
    code = ("import sys; sys.path[:0] = ['.', 'tests']\nimport numpy as np\nfrom test_hip_launch_thread import HipBackend, rolled\n"
            "be = HipBackend(0); y, want = rolled(be, 100)\nassert np.array_equal(be.to_numpy(y), want); print('same')")
    r = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, CG_LAUNCH_THREAD="0"), cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                       capture_output=True, text=True, timeout=100)
    assert r.stdout.endswith("same\n"), r.stderr
