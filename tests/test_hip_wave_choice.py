"""Decode steps of models with experts where their kernels' lanes end: the choice of experts by a wave (up to 64, groups of a power of two
members, equal scores) and beside it, and heads whose lanes, pairs of the rotation and rounds of waves are not whole ones; against float64 with the
tolerances of the blocks' other tests."""
import numpy as np
import pytest

import block_cases as C

pytestmark = pytest.mark.gpu


# experts, top, groups, keep
@pytest.mark.parametrize("count,top,groups,keep", [(64, 8, 1, 1), (64, 8, 8, 3), (63, 7, 1, 1), (33, 4, 33, 9), (64, 3, 2, 1), (64, 5, 1, 1), (48, 6, 3, 2), (60, 8, 4, 2), (65, 8, 1, 1), (128, 8, 4, 2)])
@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_choice(hip, count, top, groups, keep, dt):
    def ties(t): # (the first of equal ones counts)
        t["logits"][:] = np.round(t["logits"])
        t["correction"][:] = 0.0

    case = (2, 72, count, top, groups, keep, 24, 48, dt)
    C.run_experts(hip, case)
    C.run_experts(hip, case, seed=5, change=ties)


# heads, KV heads, head size, value size, turned columns
@pytest.mark.parametrize("heads,kv,dim,vdim,rot", [(32, 16, 128, 32, 6), (32, 8, 68, 64, 34), (20, 5, 36, 20, 36), (9, 3, 64, 12, 2), (40, 40, 32, 12, 30), (6, 2, 4, 4, 4)])
def test_heads(hip, heads, kv, dim, vdim, rot):
    o, rng = C.turned(heads, kv, dim, vdim, rot), np.random.default_rng(dim)
    C.check_attention(hip, C.attention_case(rng, 2, 78, o, False, True), o, [70, 1, 1, 3, 1, 2], tol=6e-5)
