"""The experts' f32 products of a prompt with values that bfloat16 pieces do not hold, in some tokens' rows and in some of an expert's
columns: both tile heights, both products; what lies beside such values in a tile keeps its accuracy."""
import numpy as np
import pytest

import block_cases as C
import lufatar_reference as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,count,top", [(300, 16, 2), (300, 4, 2), (1100, 8, 3)])
@pytest.mark.parametrize("where", ["tokens", "columns", "both", "infinity"])
def test_values_beyond_the_pieces(hip, rows, count, top, where):
    rng = np.random.default_rng(rows + count)
    width, ff, limit = 136, 88, 1.2
    t = C.expert_case(rng, rows, width, count, ff, "f32")
    far, lost = np.float32(2.0 ** 100), []
    if where in ("tokens", "both"):
        t["h"][0, [0, 7, rows // 2, rows - 1]] *= far         # (both factors of an activation are clamped)
    if where in ("columns", "both"):
        t["down"][1, [0, 33, 64, width - 1]] *= far
        t["down"][count - 1, 5] *= far
    if where == "infinity":
        lost = [3, rows - 2]
        t["h"][0, lost, 11] = np.inf
    keep = np.setdiff1d(np.arange(rows), lost)
    h, s = t["h"][0].astype(np.float64), L.sigmoid(t["logits"][0].astype(np.float64))
    want, bound = np.zeros((rows, width)), np.zeros((rows, width))
    for r in keep:
        for e in L.chosen_experts(s[r] + t["correction"], top, 2, 2):
            gate, up = t["gate_up"][e].astype(np.float64)
            down = t["down"][e].astype(np.float64)
            g, u = np.minimum(h[r] @ gate.T, limit), np.clip(h[r] @ up.T, -limit, limit)
            act = g * L.sigmoid(1.702 * g) * (u + 1.0)
            want[r] += s[r, e] * (act @ down.T)
            # the tolerance of the experts' other tests, here of the sum of magnitudes behind each value
            bound[r] += s[r, e] * 3e-5 * (np.abs(act) @ np.abs(down).T)
    ex = {n: hip.from_numpy(t[n]) for n in ("logits", "correction", "h")}
    ex.update({n: C.weight(hip, t[n], "f32") for n in ("gate_up", "down")})
    x = np.zeros((1, rows, width), np.float32)
    got = hip.to_numpy(hip.block_residual(hip.from_numpy(x), [], scale=1.0, experts=ex, top=top, groups=2, keep=2, limit=limit, slope=1.702))[0]
    err = np.abs(got - want)[keep] / bound[keep]
    print(where, "error / bound: max %.4f" % err.max(), flush=True)
    assert (err <= 1.0).all()
