"""Attention of a few tokens behind a cache: the kernel that takes all keys of 16 columns at once, and the one by segments of keys beside
it, at the edges of their tiles, against the plain statement."""
import numpy as np
import pytest

import block_cases as C

pytestmark = pytest.mark.gpu

# heads, kv heads, widths of keys and values, window, batch, portions, options: keys around a segment (128) and a pass (1024), columns that are not whole pieces of 16, one to
# eleven heads per kv head, more heads than are in flight (16), widths beyond the loads in flight (128), more segments than lanes (64)
CASES = [(2, 2, 16, 16, 0, 1, [126, 1, 1, 1, 1], {}), (4, 2, 132, 20, 0, 1, [255, 1, 1, 2], {}), (8, 1, 8, 36, 0, 1, [1021, 1, 1, 1, 1, 1], {}), (20, 5, 12, 16, 0, 2, [300, 1, 3, 8], {}),
         (34, 2, 8, 12, 0, 1, [140, 1, 2], {}), (11, 1, 8, 4, 0, 1, [130, 1, 1], {}), (6, 2, 16, 20, 130, 1, [200, 1, 1, 7], {}), (16, 8, 128, 128, 0, 1, [513, 1, 1], {}),
         (8, 4, 16, 32, 0, 1, [257, 1, 1], {"zero_sink": 1, "distance_bias": 0, "temp_every": 0}), (1, 1, 4, 4, 0, 1, [8190, 1, 1, 1, 1], {}), (8, 8, 16, 16, 0, 8, [129, 1, 8], {}),
         (16, 16, 8, 80, 0, 8, [129, 1, 8], {}), (4, 4, 12, 16, 0, 1, [1] * 5, {})]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c[:6])))
@pytest.mark.parametrize("talk", [True, False])
def test_columns(hip, case, talk):
    heads, kv_heads, dim, vdim, window, B, portions, extra = case
    rng = np.random.default_rng(sum(case[:5]))
    o = C.options(heads, kv_heads, dim, vdim, window, **extra)
    C.check_attention(hip, C.attention_case(rng, B, sum(portions), o, True, talk), o, portions, tol=6e-5)


def test_weights_beyond_32_bits(hip):
    """Scores thousands apart, all of a segment far below the others: its exponentials are taken behind its own maximum, and weigh nothing."""
    o = C.options(2, 1, 4, 16, 0, distance_bias=0, temp_every=0, scale=1.0)
    rng = np.random.default_rng(3)
    t = C.attention_case(rng, 1, 300, o, norms=False)
    t["k"][0, :128] -= 2000.0
    t["q"] = np.abs(t["q"])
    C.check_attention(hip, t, o, [297, 1, 1, 1], tol=2e-3)  # (scores of 2^12 in 24 bits: 2^-12 of a weight)
