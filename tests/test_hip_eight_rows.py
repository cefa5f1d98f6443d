"""Steps of five to eight sequences: the products' kernels with a second group of four rows (norms in the loads, residual sums with
their row sums, gated pairs, rotary embedding and cache rows in the store, normed heads), against the float64 model."""
import numpy as np
import pytest

import np_models
from catgrad_amd.runner import LlmConfig, Session
from model_cases import params_of, prompt_of

pytestmark = pytest.mark.gpu

# (hidden, heads, kv heads, feed-forward, head size, kind): whole and ragged chunks of k of 1024 and 2048, one chunk and several,
# outputs wide enough for the eight-column kernel and not, normed heads
SHAPES = {
    "ragged_short": ("llama", 576, 9, 3, 1536, 0),
    "one_short_chunk": ("llama", 1024, 16, 4, 3072, 0),
    "eight_columns": ("llama", 2048, 32, 8, 4096, 0),
    "ragged_long": ("llama", 2304, 18, 6, 1024, 0),
    "short_chunks": ("llama", 3072, 24, 8, 1028, 0),
    "normed_heads": ("qwen3", 1024, 16, 8, 3072, 128),
    "normed_heads_64": ("qwen3", 1536, 12, 4, 768, 64),
}


@pytest.fixture(scope="module")
def session():
    return Session()


@pytest.mark.parametrize("rows", [5, 8])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_steps_of_five_to_eight_rows(session, shape, rows):
    check(session, SHAPES[shape], rows)


# last chunks that end inside a run of 64 values of k, with no chunk before them and with one
ENDS = {"hidden_580": ("qwen3", 580, 9, 3, 1156, 64), "hidden_1156": ("llama", 1156, 17, 17, 580, 0), "hidden_3332": ("qwen3", 3332, 8, 4, 2308, 128)}


@pytest.mark.parametrize("rows", [1, 4, 7])
@pytest.mark.parametrize("shape", ["ragged_short", "ragged_long", "short_chunks", *ENDS])
def test_steps_with_ragged_chunks(session, shape, rows):
    check(session, ENDS.get(shape) or SHAPES[shape], rows)


# every number of trips that a last chunk can have, behind no chunk and behind one: heads of 64
TRIPS = {f"hidden_{h}": ("llama", h, 8, 2, h + 4, 64) for h in (264, 772, 1796, 2564, 2820)}


@pytest.mark.parametrize("rows", [1, 4, 8])
@pytest.mark.parametrize("shape", list(TRIPS))
def test_steps_with_every_last_chunk(session, shape, rows):
    check(session, TRIPS[shape], rows)


@pytest.mark.parametrize("K", [260, 512, 516, 768, 772, 1020, 1024, 1028, 1284, 1536, 1540, 1796, 2044, 2048, 2052, 2304, 2560, 2564, 2816, 2820, 3076, 3332, 4100])
def test_products_of_every_last_chunk(hip, K):
    """Alone, two and three in a launch, with a residual sum; columns for one and for two groups of four a workgroup.  Whole numbers: every order of
    summation gives the same."""
    rng = np.random.default_rng(K)
    for N in (2052, 4100, 8196):
        w = rng.integers(-3, 4, (3, N, K)).astype(np.float32)
        tw = [hip.from_numpy(a) for a in w]
        for rows in (1, 4, 5, 8):
            x, r = rng.integers(-3, 4, (1, rows, K)).astype(np.float32), rng.integers(-9, 10, (1, rows, N)).astype(np.float32)
            tx, want = hip.from_numpy(x), [x[0] @ a.T for a in w]

            def product(i):
                return hip.matmul(tx, hip.broadcast(hip.transpose(tw[i], 0, 1), (1, K, N)).move())

            np.testing.assert_array_equal(hip.to_numpy(product(0))[0], want[0])
            for n in (2, 3):
                for i, y in enumerate([product(i) for i in range(n)]):
                    np.testing.assert_array_equal(hip.to_numpy(y)[0], want[i])
            np.testing.assert_array_equal(hip.to_numpy(hip.add(product(1).move(), hip.from_numpy(r)))[0], want[1] + r[0])


def check(session, shape, rows):
    arch, hidden, heads, kv, ff, hd = shape
    cfg = LlmConfig(arch, hidden, 2, heads, kv, ff, 521, head_dim=hd, rms_norm_eps=1e-5, rope_theta=10000.0, tie_word_embeddings=True)
    params = params_of(cfg, seed=rows, scale=1.5)
    rng = np.random.default_rng(7)
    for name, w in params.items():  # gains that tell columns apart
        if w.ndim == 1:
            params[name] = (1.0 + 0.3 * rng.standard_normal(w.shape)).astype(np.float32)
    session.load_model(cfg, params=params.items())
    # one run of that many rows: logits.  A sum of n products is off by n 2^-24 of its magnitudes at most, by sqrt(n) of that in the
    # mean; the longest here is 4096, there are ten in a row
    prompt = prompt_of(cfg, rows, 1, seed=rows + 1)
    _, got = session.forward(prompt, max_positions=4)
    want = np_models.llm_logits(cfg, params, prompt)
    assert np.abs(got - want).max() <= 10 * 4 * 4096 ** 0.5 * 2.0 ** -24 * np.abs(want).max()
    # and greedy steps behind it: every token is the float64 model's choice for the same sequence so far
    steps = 6
    tokens, _ = session.generate(prompt, steps)
    seq = np.concatenate([prompt, tokens[:-1].T], axis=1)
    want = np_models.llm_logits(cfg, params, seq)
    chosen = np.take_along_axis(want, tokens.T[:, :, None].astype(np.int64), -1)[..., 0]
    assert (want.max(-1) - chosen <= 10 * 4 * 4096 ** 0.5 * 2.0 ** -24 * np.abs(want).max()).all()
