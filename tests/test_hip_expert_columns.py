"""The experts' first products for a few rows with several columns per wave: one after the other with the next one on its way, and in halves
where a column is eight pieces long; alone against the plain statement, beside attention against a launch of their own."""
import numpy as np
import pytest

import block_cases as C

pytestmark = pytest.mark.gpu

# rows, width, experts, top, groups, keep, ff, K, dtype: one to eight pieces of 256 or 512 values and beyond, two to four columns per wave (columns / 8192), the last
# workgroup with fewer
CASES = [(8, 256, 4, 2, 2, 1, 1304, 0, "f32"), (8, 504, 4, 2, 2, 1, 1544, 0, "f32"), (8, 1024, 2, 2, 1, 1, 2056, 0, "f32"), (8, 2048, 2, 2, 1, 1, 1544, 0, "f32"), (8, 2056, 2, 2, 1, 1, 1304, 0, "f32"),
         (8, 512, 4, 2, 2, 1, 1544, 0, "bf16"), (8, 1000, 2, 2, 1, 1, 1304, 0, "bf16"), (7, 2048, 2, 2, 1, 1, 1784, 0, "bf16"), (8, 4096, 2, 2, 1, 1, 1544, 0, "bf16")]


@pytest.mark.parametrize("case", CASES, ids=str)
def test_columns(hip, case):
    C.run_experts(hip, case)


# width, experts' columns, dtype: 24 workgroups of attention leave 744 to the experts, with one to three columns per wave
@pytest.mark.parametrize("width,ff,dt", [(512, 1480, "f32"), (1024, 1496, "f32"), (2048, 3000, "bf16"), (4096, 4000, "bf16")], ids=str)
def test_beside_attention(hip, width, ff, dt):
    def run(wait):
        be, rng = hip, np.random.default_rng(ff)
        heads, kv_heads, dim, count = 8, 4, 64, 2
        o = C.turned(heads, kv_heads, dim, dim, 16)
        t = C.attention_case(rng, 1, 1, o, norms=False)
        caches = [be.from_numpy(rng.standard_normal((1, kv_heads, 90, dim)).astype(np.float32)) for _ in range(2)]
        e = C.expert_case(rng, 1, width, count, ff, dt)
        ex = {n: be.from_numpy(e[n].reshape((1, 1, -1) if n == "logits" else e[n].shape)) for n in ("logits", "correction")}
        h = be.from_numpy(e["h"].reshape(1, 1, width))
        ex["h"] = h if dt == "f32" else be.cast(h, C.BF16)
        ex.update({n: C.weight(be, e[n], dt) for n in ("gate_up", "down")})
        w = C.weight(be, C.bf16(rng.standard_normal((width, heads * dim)) * 0.04), dt)
        x, tensors = be.from_numpy(rng.standard_normal((1, 1, width)).astype(np.float32)), {n: be.from_numpy(t[n]) for n in ("q", "k", "v", "talk")}
        for v in list(ex.values()) + [w, x]:
            be.realize(v)
        y, kc, vc = be.block_attention({**tensors, "k_cache": caches[0].move(), "v_cache": caches[1].move()}, position=90, **o)
        if wait:
            be.sync()
        out = be.block_residual(x, [{"y": y.move(), "w": w}], scale=0.4, experts=ex, top=2, groups=1, keep=1, limit=1.2, slope=1.702)
        return [be.to_numpy(a) for a in (out, kc, vc)]
    for a, b in zip(run(False), run(True)):
        np.testing.assert_array_equal(a, b)
