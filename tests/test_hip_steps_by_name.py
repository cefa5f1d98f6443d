"""Decode steps of models with experts where their kernels' lanes end: the choice of experts by a wave (up to 64, groups of a power of two
members, equal scores) and beside it, pieces of the experts' second products, and heads whose lanes, pairs of the rotation and rounds of waves
are not whole ones; against float64 with the tolerances of the blocks' other tests."""
import numpy as np
import pytest

import block_cases as C
import kernel_names
from backends import backend_with_env

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def narrow():
    """Stores bfloat16 tensors of any size as such (others: from 65536 elements on)."""
    be = backend_with_env(CG_NARROW_FROM="2")
    yield be
    be.close()


# experts, top, groups, keep
@pytest.mark.parametrize("count,top,groups,keep", [(64, 8, 1, 1), (64, 8, 8, 3), (63, 7, 1, 1), (33, 4, 33, 9), (64, 3, 2, 1), (64, 5, 1, 1), (48, 6, 3, 2), (60, 8, 4, 2), (65, 8, 1, 1), (128, 8, 4, 2)])
@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_choice(narrow, count, top, groups, keep, dt):
    def ties(t): # (the first of equal ones counts)
        t["logits"][:] = np.round(t["logits"])
        t["correction"][:] = 0.0

    case = (2, 72, count, top, groups, keep, 24, 48, dt)
    C.run_experts(narrow, case, behind=8)
    C.run_experts(narrow, case, seed=5, change=ties, behind=8)


# choices and pieces of the output product, and how many pieces a wave takes at a time (each choice is one piece here)
PIECES = [(1, 0, 1), (4, 0, 1), (5, 0, 2), (8, 0, 2), (8, 1, 3), (8, 4, 3), (8, 5, 4), (8, 8, 4), (8, 9, 5), (8, 12, 5), (8, 13, 6), (8, 16, 6),
          (8, 17, 4), (8, 24, 4), (8, 25, 5), (8, 40, 6), (8, 41, 5)]  # two rounds, three


def pieces(be, top, more, dt):
    span = 256 if dt == "f32" else 512
    C.run_experts(be, (2, 40, 16, top, 1, 1, 64, more * span - 8 * (more > 1), dt), behind=8)


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("top,more,at_once", PIECES)
def test_pieces(narrow, top, more, at_once, dt):
    pieces(narrow, top, more, dt)


# heads, KV heads, head size, value size, turned columns
HEADS = [(32, 16, 128, 32, 6), (32, 8, 68, 64, 34), (20, 5, 36, 20, 36), (9, 3, 64, 12, 2), (40, 40, 32, 12, 30), (6, 2, 4, 4, 4)]


def heads_of(be, heads, kv, dim, vdim, rot):
    o, rng = C.turned(heads, kv, dim, vdim, rot), np.random.default_rng(dim)
    C.check_attention(be, C.attention_case(rng, 2, 78, o, False, True), o, [70, 1, 1, 3, 1, 2], tol=6e-5, behind=8)


@pytest.mark.parametrize("heads,kv,dim,vdim,rot", HEADS)
def test_heads(hip, heads, kv, dim, vdim, rot):
    heads_of(hip, heads, kv, dim, vdim, rot)


@pytest.mark.parametrize("name", list(C.MIXED))
def test_mixed_scores_in_steps(hip, name):
    """The other tests' cases on rows at 16 bytes, which portions of a few tokens have kernels of their own for."""
    C.run_mixed_case(hip, name, behind=8)


@pytest.mark.parametrize("heads,kv,dim,vdim", [(16, 8, 128, 128), (8, 2, 64, 64), (4, 4, 32, 32), (16, 2, 128, 64)])
def test_many_chunks_a_workgroup(hip, heads, kv, dim, vdim):
    """Segments of several chunks, whose values come behind the first one's: 8 x 8 new tokens behind many cached ones."""
    o, rng = C.turned(heads, kv, dim, vdim, 32, norm_eps=1e-3), np.random.default_rng(dim)
    S = 700
    t = C.attention_case(rng, 8, S + 8, o, False, True)
    C.check_attention(hip, t, o, [S, 8], tol=6e-5, behind=8)


def test_which_kernels(tmp_path):
    kernel_names.run(tmp_path, r"""
import re
import test_hip_steps_by_name as T
be = T.backend_with_env(CG_NARROW_FROM="2")


def count(names, pattern):
    return sum(bool(re.search(pattern, n)) for n in names)


for dt in ("f32", "bf16"):
    for top, more, at_once in T.PIECES:
        names = launches(be, T.pieces, be, top, more, dt)
        print(dt, top, more, at_once, flush=True)
        assert count(names, "expert_first_kernelILb%dELb1E" % (dt == "bf16")) == 1, names
        assert count(names, "expert_second_kernelILb%dELb1ELi%dE" % (dt == "bf16", at_once)) == 1, names
for sizes in T.HEADS:
    names = launches(be, T.heads_of, be, *sizes)
    print(sizes, flush=True)
    assert count(names, "attention_mixed_step_kernel") == 5, names
for case in ((16, 8, 128, 128), (16, 2, 128, 64)):
    names = launches(be, T.test_many_chunks_a_workgroup, be, *case)
    print(case, flush=True)
    assert count(names, "attention_mixed_step_kernel") == 1, names
print("done", flush=True)
""")
