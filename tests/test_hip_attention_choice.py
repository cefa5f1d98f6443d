"""A decode step's attention around the lengths where rows or segments of the cache are the quicker way, both merged from up to 256 segments,
against the closed form; and without the scratch memory of the segments, which are then left."""
import os
import subprocess
import sys

import numpy as np
import pytest

import kernel_names
import test_hip_no_room
from cases import _np_decode_attention, decode_attention_ops, f32

pytestmark = pytest.mark.gpu

# sequences, KV heads, query rows per KV head, head size, positions on either side of the choice; the last ones: 64, 65 and 256 segments, five to eight rows per
# KV head, more query rows than compute units
CASES = [(1, 8, 2, 128, (380, 420, 511, 512)), (1, 8, 4, 64, (1000, 1060, 1300)), (1, 3, 3, 64, (767, 780, 1025)), (4, 8, 2, 128, (500, 640, 1024)), (4, 8, 4, 64, (1536, 2047, 4096)),
         (1, 1, 2, 128, (4096, 4097)), (1, 1, 3, 64, (4095, 4160, 16384)), (1, 2, 8, 128, (500, 700)), (3, 2, 5, 64, (900, 1400)), (9, 8, 4, 64, (1023, 1024, 1100))]


@pytest.mark.parametrize("B,kvh,rep,hd,T", [(*c[:4], T) for c in CASES for T in c[4]])
def test_choice(hip, B, kvh, rep, hd, T):
    q, k, v = f32(400 + T, (B, kvh * rep, 1, hd)), f32(401 + T, (B, kvh, T, hd)), f32(402 + T, (B, kvh, T, hd))
    got = hip.to_numpy(decode_attention_ops(hip, hip.from_numpy(q), hip.from_numpy(k), hip.from_numpy(v), rep))
    np.testing.assert_allclose(got, _np_decode_attention(q, k, v, rep), rtol=1e-4, atol=1e-5)


# the last length of rows and the first of segments
EDGES = [(1, 8, 2, 128, 485), (1, 8, 4, 64, 1126), (1, 3, 3, 64, 969), (4, 8, 2, 128, 644), (4, 8, 4, 64, 1646), (1, 2, 8, 128, 680), (3, 2, 5, 64, 1360)]


@pytest.mark.parametrize("B,kvh,rep,hd,T", [(*c[:4], c[4] + d) for c in EDGES for d in (-1, 0)])
def test_edges(hip, B, kvh, rep, hd, T):
    test_choice(hip, B, kvh, rep, hd, T)


def test_which_is_chosen(tmp_path):
    kernel_names.run(tmp_path, r"""
from catgrad_amd import HipBackend
from cases import decode_attention_ops, f32
from test_hip_attention_choice import EDGES
be = HipBackend(0)
for B, kvh, rep, hd, first in EDGES:
    for T, want in ((first - 1, "decode_attention_row_kernel"), (first, "decode_attention_seg_kernel")):
        x = [be.from_numpy(f32(1, s)) for s in ((B, kvh * rep, 1, hd), (B, kvh, T, hd), (B, kvh, T, hd))]
        names = [n for n in launches(be, lambda: be.realize(decode_attention_ops(be, *x, rep))) if "decode_attention" in n]
        assert want in names[0] and len(names) == (2 if "seg" in want else 1), (B, kvh, rep, hd, T, names)
print("done", flush=True)
""")


PROGRAM = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)        # before the library: its requests come here first
shim.refuse.argtypes = [ctypes.c_size_t] * 2
sys.path.insert(0, sys.argv[2])
import numpy as np
from cases import _np_decode_attention, decode_attention_ops, f32
from catgrad_amd import HipBackend
be = HipBackend(0)
for B, kvh, rep, hd, T, asked in ((1, 8, 2, 128, 1000, True), (2, 8, 4, 64, 4000, True), (1, 8, 2, 128, 300, False)):
    a = [f32(400 + T, (B, kvh * rep, 1, hd)), f32(401 + T, (B, kvh, T, hd)), f32(402 + T, (B, kvh, T, hd))]
    want = _np_decode_attention(*a, rep)
    x = [be.from_numpy(t) for t in a]
    be.pool_trim()
    shim.refuse(50_000, 16 << 20)
    y = decode_attention_ops(be, *x, rep)
    be.realize(y)
    be.sync()
    seen = shim.count()
    shim.refuse(1, 0)
    print(B, kvh, rep, hd, T, "requests refused:", seen, flush=True)
    assert bool(seen) == asked
    np.testing.assert_allclose(be.to_numpy(y), want, rtol=1e-4, atol=1e-5)
print("done", flush=True)
"""


def test_without_scratch_memory(tmp_path):
    here = os.path.dirname(os.path.abspath(__file__))
    (tmp_path / "shim.c").write_text(test_hip_no_room.SHIM)
    (tmp_path / "program.py").write_text(PROGRAM)
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", str(tmp_path / "shim.so"), str(tmp_path / "shim.c"), "-ldl"])
    env = dict(os.environ, PYTHONPATH=os.path.dirname(here))
    r = subprocess.run([sys.executable, str(tmp_path / "program.py"), str(tmp_path / "shim.so"), here], env=env, capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0 and r.stdout.endswith("done\n")
