"""A backend's launches go through a thread of its own when there are many between two waits of the host: whatever else is put on the
stream, allocated or given back in between stays in order, on every backend and from every thread."""
import os
import subprocess
import sys
import threading

import numpy as np
import pytest

from catgrad_amd import HipBackend

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


def test_threads_and_backends():
    shared, wrong = HipBackend(0), []

    def work(be):
        for n in (5, 50, 100):
            y, want = rolled(be, n)
            wrong.extend([n] if not np.array_equal(be.to_numpy(y), want) else [])

    t = [threading.Thread(target=work, args=(shared if i % 2 else HipBackend(0),)) for i in range(6)]
    for x in t:
        x.start()
    for x in t:
        x.join()
    assert not wrong


def test_backend_dropped_with_launches_on_their_way():
    for _ in range(5):
        be = HipBackend(0)
        rolled(be, 100)
        del be


def test_without_the_thread():
    code = ("import sys; sys.path[:0] = ['.', 'tests']\nimport numpy as np\nfrom test_hip_launch_thread import HipBackend, rolled\n"
            "be = HipBackend(0); y, want = rolled(be, 100)\nassert np.array_equal(be.to_numpy(y), want); print('same')")
    r = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, CG_LAUNCH_THREAD="0"), cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                       capture_output=True, text=True, timeout=100)
    assert r.stdout.endswith("same\n"), r.stderr
