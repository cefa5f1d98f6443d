"""One token of the gated delta rule behind a state (delta_token_kernel), at the edges of its rows, columns and ranks, and beside them,
against float64: the tolerance is the other portions'."""
import numpy as np
import pytest

import block_cases as C

pytestmark = pytest.mark.gpu


# (heads, KV heads, key channels, value channels, ranks)
@pytest.mark.parametrize("heads,kv,dim,vdim,ranks", [
    (1, 1, 1, 4, (4, 4)), (2, 1, 31, 60, (64, 60)), (4, 2, 32, 64, (8, 64)), (2, 2, 128, 64, (68, 4)),  # four lanes' sixteenths of a row
    (2, 1, 127, 68, (64, 12)), (3, 3, 65, 128, (4, 128)), (2, 1, 128, 124, (72, 128)),  # eighths
    (2, 1, 129, 64, (8, 8)), (2, 1, 64, 132, (8, 8)), (2, 1, 64, 62, (8, 8)), (2, 2, 16, 16, (132, 8)), (2, 2, 16, 16, (8, 10)),  # the general kernel's
])
def test_one_token_behind_a_state(hip, heads, kv, dim, vdim, ranks):
    rng = np.random.default_rng(dim + 1000 * vdim)
    o = C.delta_options(heads, kv, dim, vdim)
    C.check_delta(hip, C.delta_case(rng, 2, 24, o, 4, *ranks), o, [19, 1, 1, 2, 1])
    C.check_delta(hip, C.delta_case(rng, 1, 4, o, 4, *ranks, decay_at=6.0), o, [1, 1, 1, 1])
