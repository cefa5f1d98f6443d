"""The work whose speed matters here, as cases that can be timed and checked.

A case is what a program using this package does between having its inputs and having its results, through the public entry
points: `Session` (whole models on the host driver) and `HipBackend` (one operation at a time).  Six kinds:

  request     one sequence: `Session.step` over a prompt (whole, or in portions), then token by token over ids that the program
              already has (a replayed trace, a scored continuation, a constrained output); the logits of the wanted places come back
  batch       several prompts of one length at once, `Session.forward_rows`: the arg-max of every position and some rows' logits
  generate    greedy generation for a batch of short prompts, `Session.generate`
  mlp         a small feed-forward classifier, `Session.mlp`
  narrow      a gated feed-forward and a classifier over 16-bit or 8-bit tensors, operation by operation through `HipBackend`
  statistics  the log-sum-exp and the arg-max of rows of scores, operation by operation

Models have the sizes of the benchmark configurations and random weights.  A program loads a model once and keeps it, so a
process keeps one session per model; what differs from state to state is the tokens.  `exact` states every kind in 64-bit
torch, from the same weights and inputs and without the package's kernels or host driver."""
import math
import zlib

import numpy as np
import torch

from catgrad_amd import HipBackend, _abi as A
from catgrad_amd import loretar, lufatar
from catgrad_amd.runner import LLAMA_3_2_1B, QWEN3_0_6B, SMOLLM2_135M, Session

# ------------------------------------------------------------------------------------------------ models

DENSE = {"smollm2": SMOLLM2_135M, "qwen3": QWEN3_0_6B, "llama": LLAMA_3_2_1B}


def _loretar(width, ff, vocab, runs, at, de):
    """Half of the layer runs attend within a window of 1024, half are a delta rule; the middle half of them runs twice."""
    once = runs // 4
    n = 2 * once + (runs - 2 * once) // 2
    layers = [loretar.attention_layer(*at, 1024, ff) if i % 2 else loretar.delta_layer(*de, ff) for i in range(n)]
    return loretar.config_of(layers, vocab, width, loop={"start": once, "stop": n - once, "times": 2})


def _lufatar(width, ff, vocab, runs, at, base):
    """Every layer run attends; the feed-forward is 8 of 32 experts; the middle half of the layer runs happens twice."""
    once = runs // 4
    n = 2 * once + (runs - 2 * once) // 2
    moe = lufatar.experts(32, 8, ff, groups=4, keep=2, limit=7.0)
    layers = [lufatar.attention_layer(*at, moe, rot=64, base=base) for _ in range(n)]
    return lufatar.config_of(layers, vocab, width, loop={"start": once, "stop": n - once, "times": 2}, groups=4, mult=0.5, taps=4, side=64,
                             buckets=65521, mul_prev=7919, mul_cur=104729)


BLOCKS = {
    "loretar_small": _loretar(1024, 3072, 151936, 28, (16, 8, 128, 128), (8, 8, 128, 128)),
    "loretar_large": _loretar(2048, 8192, 128256, 16, (32, 8, 64, 64), (16, 16, 128, 128)),
    "lufatar_small": _lufatar(1024, 384, 151936, 28, (16, 8, 128, 128), 1000000.0),
    "lufatar_large": _lufatar(2048, 1024, 128256, 16, (32, 8, 64, 64), 500000.0),
}


def _shapes(model):
    if model in DENSE:
        return DENSE[model].param_shapes()
    return loretar.param_shapes(BLOCKS[model], 64) if model.startswith("loretar") else lufatar.param_shapes(BLOCKS[model])


def _weight(model, name, shape, dtype):
    """A weight tensor on the GPU in 32 bits, with values that a file of `dtype` can hold.  Scales as in the package's own random
    weights: matrices keep their input's scale (0.02 in the dense models), norms scatter around one (dense: are one)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(zlib.crc32(f"{model}/{name}".encode()))
    n = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    if model in DENSE:
        n = torch.ones_like(n) if len(shape) == 1 else n * 0.02
    elif name.endswith(("norm", "norm1", "norm2")):
        n = 1.0 + 0.2 * n
    elif name.endswith(".talk"):
        n = torch.eye(shape[0], device="cuda") + 0.3 * n
    elif name.endswith(".A_log"):
        n = 0.5 * n
    elif name.endswith(".dt_bias"):
        n = n - 3.0
    elif name.endswith(".mlp.act"):
        n = 0.5 + 0.2 * n
    elif name.endswith((".canon1", ".canon2")):
        n = n * (0.5 * shape[1] ** -0.5)
    elif name in ("embed", "bigram", "side.embed"):
        pass
    elif len(shape) == 2 and name != "loop.step":
        n = n * shape[1] ** -0.5
    elif name.endswith(".correction") and dtype == "bfloat16":
        # so far apart that no rounding changes a choice: with choices on the edge, models at this precision answer differently
        # whenever a sum is taken in another order (the 32-bit weights choose by the tokens)
        n = 2.5 * 2.0 ** torch.argsort(n).float() - 60.0
    else:
        n = 0.2 * n
    return n.bfloat16().float() if dtype == "bfloat16" else n


_sessions, _backend, _weights, _staging = {}, [], {}, []


def _host(t):
    """A 32-bit GPU tensor's values as a numpy array that the next call overwrites (pinned memory: copies run at full speed)."""
    if not _staging or _staging[0].numel() < t.numel():
        _staging[:] = [torch.empty(max(t.numel(), 1 << 20), dtype=torch.float32, pin_memory=True)]
    out = _staging[0][: t.numel()]
    out.copy_(t.reshape(-1))
    return out.numpy().reshape(tuple(t.shape))


def _session(model, dtype):
    """The session a program keeps for a model."""
    if (model, dtype) not in _sessions:
        s = Session()
        if model in DENSE:
            s.clear_params()
            for name, shape in _shapes(model):
                s.set_param(name, _host(_weight(model, name, shape, dtype)))
            s.set_config(DENSE[model])
        else:
            s.load_config(BLOCKS[model], dtype)
            for name, shape in _shapes(model):
                s.set_param(name, _host(_weight(model, name, shape, dtype)))
        s.sync()
        _sessions[model, dtype] = s
    return _sessions[model, dtype]


def _ops():
    if not _backend:
        _backend.append(HipBackend(0))
    return _backend[0]


def _vocab(model):
    return DENSE[model].vocab_size if model in DENSE else BLOCKS[model]["vocab"]


# ------------------------------------------------------------------------------------------------ the cases

def listed():
    return [
        # the smallest model there is: a classifier called on 64 rows, where launches and the way to the device count
        {"name": "mlp_64", "kind": "mlp", "rows": 64, "inputs": 256, "hidden": 512, "outputs": 10},
        # scoring of ready logits: two passes over memory, no products
        {"name": "statistics_4096x8192", "kind": "statistics", "dtype": "float32", "rows": 4096, "cols": 8192},
        # a feed-forward on reduced-precision tensors, at the widths of the 1B-size models: a full batch, and a ragged smaller one
        {"name": "narrow_bf16_8192", "kind": "narrow", "dtype": "bfloat16", "rows": 8192, "width": 2048, "hidden": 8192, "classes": 16},
        {"name": "narrow_fp8_1500", "kind": "narrow", "dtype": "float8", "rows": 1500, "width": 2048, "hidden": 8192, "classes": 16},
        # a small dense model: prompt and a short answer
        {"name": "smollm2_512_16", "kind": "request", "model": "smollm2", "dtype": "float32", "prompt": 512, "portion": 0, "decode": 16},
        # a mid-size dense model with normed heads: decoding behind a longer prompt
        {"name": "qwen3_1024_48", "kind": "request", "model": "qwen3", "dtype": "float32", "prompt": 1024, "portion": 0, "decode": 48},
        # the largest: four long prompts at once
        {"name": "llama_4x2048", "kind": "batch", "model": "llama", "batch": 4, "prompt": 2048, "rows": 16},
        # greedy generation for four short prompts: weights streamed once a step
        {"name": "llama_generate_4x8_48", "kind": "generate", "model": "llama", "batch": 4, "prompt": 8, "decode": 48},
        # a recurrent / attention hybrid with bfloat16 weights: a long prompt in two portions
        {"name": "loretar_bf16_2048", "kind": "request", "model": "loretar_large", "dtype": "bfloat16", "prompt": 2048, "portion": 1024, "decode": 0},
        # the same design in 32 bits: a ragged prompt and an answer
        {"name": "loretar_f32_777_32", "kind": "request", "model": "loretar_small", "dtype": "float32", "prompt": 777, "portion": 0, "decode": 32},
        # experts with bfloat16 weights: a ragged prompt and an answer
        {"name": "lufatar_bf16_300_32", "kind": "request", "model": "lufatar_small", "dtype": "bfloat16", "prompt": 300, "portion": 0, "decode": 32},
        # experts in 32 bits: two prompts at once
        {"name": "lufatar_f32_2x1024", "kind": "batch", "model": "lufatar_large", "batch": 2, "prompt": 1024, "rows": 16},
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, evenly over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    most = 2.3e13  # flops of the largest listed case
    while True:
        kind = rng.choice(["request"] * 6 + ["batch"] * 3 + ["generate", "generate", "mlp", "narrow", "narrow", "statistics"])
        if kind == "request":
            model = rng.choice(sorted(DENSE) + sorted(BLOCKS))
            c = {"kind": kind, "model": model, "dtype": "float32" if model in DENSE else rng.choice(["float32", "bfloat16"]),
                 "prompt": _spread(rng, 1, 2048), "portion": 0, "decode": rng.choice([0, 0, rng.randint(1, 48)])}
            if rng.random() < 0.3:
                c["portion"] = rng.randint(max(1, -(-c["prompt"] // 8)), c["prompt"])
        elif kind == "batch":
            c = {"kind": kind, "model": rng.choice(sorted(DENSE) + sorted(BLOCKS)), "batch": rng.randint(1, 8), "prompt": _spread(rng, 1, 2048)}
            c["rows"] = rng.randint(1, min(16, c["batch"] * c["prompt"]))
            if c["batch"] * c["prompt"] > (8192 if c["model"] in DENSE else 4096):
                continue
        elif kind == "generate":
            c = {"kind": kind, "model": rng.choice(sorted(DENSE)), "batch": rng.randint(1, 8), "prompt": rng.randint(1, 16), "decode": rng.randint(4, 48)}
        elif kind == "mlp":
            c = {"kind": kind, "rows": _spread(rng, 1, 2048), "inputs": _spread(rng, 8, 2048), "hidden": _spread(rng, 16, 2048), "outputs": _spread(rng, 2, 512)}
        elif kind == "narrow":
            c = {"kind": kind, "dtype": rng.choice(["bfloat16", "float16", "float8"]), "rows": _spread(rng, 9, 8192), "width": _spread(rng, 64, 2048),
                 "hidden": _spread(rng, 128, 8192), "classes": rng.randint(2, 64)}
            if rng.random() < 0.7:  # widths of models are whole multiples of 64; some are odd
                c["width"], c["hidden"] = max(64, c["width"] // 64 * 64), c["hidden"] // 64 * 64
        else:
            c = {"kind": kind, "dtype": rng.choice(["float32", "float32", "bfloat16"]), "rows": _spread(rng, 1, 8192), "cols": _spread(rng, 16, 131072)}
            if c["rows"] * c["cols"] > 4096 * 8192:
                continue
        if work(c)["flops"] <= most:
            return c


# ------------------------------------------------------------------------------------------------ inputs

NARROW = {"bfloat16": (A.BF16, torch.bfloat16, torch.int16), "float16": (A.F16, torch.float16, torch.int16), "float8": (A.F8, torch.float8_e4m3fn, torch.uint8)}


def _portions(case):
    """(first token, one behind the last, wanted places in it) of every step of a request."""
    n, size = case["prompt"], case["portion"] or case["prompt"]
    out = [(a, min(a + size, n), sorted({(min(a + size, n) - a) // 2, min(a + size, n) - a - 1})) for a in range(0, n, size)]
    return out + [(n + i, n + i + 1, [0]) for i in range(case["decode"])]


def _tokens(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] == "request":
        return rng.integers(0, _vocab(case["model"]), size=case["prompt"] + case["decode"], dtype=np.uint32)
    return rng.integers(0, _vocab(case["model"]), size=(case["batch"], case["prompt"]), dtype=np.uint32)


def _wanted_rows(case, seed):
    rng = np.random.default_rng([seed, 1])
    n = case["batch"] * case["prompt"]
    return np.sort(rng.choice(n, size=min(case["rows"], n), replace=False)).astype(np.uint32)


def _tensors(case, seed):
    """The float inputs of the kinds without a model, on the GPU, in the dtype that they are given in."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)

    if case["kind"] == "mlp":
        i, h, o = case["inputs"], case["hidden"], case["outputs"]
        return {"x": normal(case["rows"], i), "mlp.l1.weight": normal(h, i) * 0.02, "mlp.l1.bias": normal(h) * 0.02,
                "mlp.l2.weight": normal(o, h) * 0.02, "mlp.l2.bias": normal(o) * 0.02}
    if case["kind"] == "narrow":
        w, h, o = case["width"], case["hidden"], case["classes"]
        t = {"x": normal(1, case["rows"], w), "gate": normal(h, w) * w ** -0.5, "up": normal(h, w) * w ** -0.5, "down": normal(w, h) * (2.0 * h ** -0.5),
             "head": normal(o, w) * w ** -0.5}
        return {k: v.to(NARROW[case["dtype"]][1]) for k, v in t.items()}
    return {"x": (normal(case["rows"], case["cols"]) * 3.0).to(torch.float32 if case["dtype"] == "float32" else torch.bfloat16)}


def _upload(be, t, dtype):
    if dtype == "float32":
        return be.ndarray_from_vec_f32(_host(t), tuple(t.shape))
    code, _, bits = NARROW[dtype]
    raw = t.view(bits).cpu().numpy()
    if code == A.F16:
        return be.ndarray_from_vec_f16(raw.view(np.float16), tuple(t.shape))
    if code == A.BF16:
        return be.ndarray_from_vec_bf16(raw.view(np.uint16), tuple(t.shape))
    return be.ndarray_from_vec_fp8(raw, tuple(t.shape))


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "kind": kind}
    if kind in ("request", "batch", "generate"):
        s["session"] = _session(case["model"], case.get("dtype", "float32"))
        s["tokens"] = _tokens(case, seed)
        if kind == "request":
            s["steps"] = [(s["tokens"][a:b].copy(), np.array(rows, dtype=np.uint32)) for a, b, rows in _portions(case)]
        elif kind == "batch":
            s["rows"] = _wanted_rows(case, seed)
    elif kind == "mlp":
        t = _tensors(case, seed)
        s["session"] = Session()
        s["x"] = t.pop("x").cpu().numpy()
        for name, w in t.items():
            s["session"].set_param(name, w.cpu().numpy())
    else:
        be = _ops()
        s["backend"] = be
        s["tensors"] = {k: _upload(be, v, case["dtype"]) for k, v in _tensors(case, seed).items()}
        be.sync()
    return s


# ------------------------------------------------------------------------------------------------ one pass

def _linear(be, x, w, batch):
    o, i = w.shape
    return be.matmul(x, be.broadcast(be.transpose(w, 0, 1), (batch, i, o)).move())


def _constant(be, value, dtype, shape):
    return be.broadcast(be.cast(be.ndarray_from_vec_f32([value], ()), dtype).move(), shape)


def run(state):
    kind, case = state["kind"], state["case"]
    if kind == "request":
        s = state["session"]
        out = [s.step(1, tokens, rows, max_positions=len(state["tokens"])) for tokens, rows in state["steps"]]
        s.end(1)
        return out
    if kind == "batch":
        ids, logits = state["session"].forward_rows(state["tokens"], state["rows"])
        return {"ids": ids, "logits": logits}
    if kind == "generate":
        tokens, _, logits = state["session"].generate(state["tokens"], case["decode"], want_logits=True)
        return {"tokens": tokens, "logits": logits}
    if kind == "mlp":
        return state["session"].mlp(state["x"], case["hidden"], case["outputs"])
    be, t = state["backend"], state["tensors"]
    if kind == "narrow":
        dtype, shape = NARROW[case["dtype"]][0], (1, case["rows"], case["hidden"])
        g, u = _linear(be, t["x"], t["gate"], 1), _linear(be, t["x"], t["up"], 1)
        e = be.exp(be.neg(g).move())
        e = be.div(g.move(), be.add(_constant(be, 1.0, dtype, shape).move(), e.move()).move())
        y = _linear(be, be.mul(e.move(), u.move()).move(), t["down"], 1)
        return be.to_numpy(be.cast(_linear(be, y.move(), t["head"], 1).move(), A.F32))
    shape = (case["rows"], case["cols"])
    x = be.cast(t["x"], A.F32)
    m = be.max(x)
    e = be.exp(be.sub(x, be.broadcast(m, shape).move()).move())
    lse = be.add(be.log(be.sum(e.move()).move()).move(), m.move())
    return {"lse": be.to_numpy(lse), "argmax": be.to_numpy(be.argmax(x.move()))}


# ------------------------------------------------------------------------------------------------ what a pass cannot do without

def _visible(first, n, window=None):
    """Pairs of positions that `n` queries from position `first` on see."""
    last = first + n
    if window is None or last <= window:
        return (first + 1 + last) * n // 2
    return sum(min(p + 1, window) for p in range(first, last))


def _matrices(model):
    """[(elements of a matrix that every token is multiplied with, how often a pass uses it, share of it that a token meets)]
    without the vocabulary's."""
    if model in DENSE:
        return [(s[0] * s[1], 1, 1.0) for n, s in _shapes(model) if len(s) == 2 and "embed_tokens" not in n and "lm_head" not in n]
    c, out = BLOCKS[model], []
    lp = c["loop"]
    for n, s in _shapes(model):
        if len(s) != 2 or n.endswith((".conv", ".talk", ".canon1", ".canon2")) or n in ("embed", "bigram", "side.embed", "loop.step", "head"):
            continue
        i = int(n[1:].split(".")[0]) if n != "loop.in" else None
        again = lp["times"] if i is None or lp["start"] <= i < lp["stop"] else 1
        r = c["layers"][i]["mlp"]["router"] if ".mlp.e" in n else None
        out.append((s[0] * s[1], again, r["top"] / r["experts"] if r else 1.0))
    return out


def _attentions(model):
    """[(query heads, key heads, dim of keys, dim of values, window, how often)]"""
    if model in DENSE:
        c = DENSE[model]
        return [(c.num_attention_heads, c.num_key_value_heads, c.hd, c.hd, None, c.num_hidden_layers)]
    c, lp, out = BLOCKS[model], BLOCKS[model]["loop"], []
    for i, l in enumerate(c["layers"]):
        m = l["mixer"]
        if l["type"] == "attention":
            out.append((m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["mask"]["size"] if "mask" in m else None, lp["times"] if lp["start"] <= i < lp["stop"] else 1))
    return out


def _pass_work(model, dtype, batch, first, n, rows):
    """One run over n new tokens of `batch` sequences behind `first` others, `rows` rows of logits."""
    width = 2 if dtype == "bfloat16" else 4
    hidden = DENSE[model].hidden_size if model in DENSE else BLOCKS[model]["width"]
    tokens, flops, read = batch * n, 0.0, 0.0
    for size, times, share in _matrices(model):
        flops += 2.0 * size * times * share * tokens
        read += width * size * times * min(1.0, share * tokens)
    for h, g, dk, dv, window, times in _attentions(model):
        flops += 2.0 * times * batch * h * (dk + dv) * _visible(first, n, window)
        read += 4.0 * times * batch * g * (dk + dv) * min(first + n, window or first + n)
    flops += 2.0 * rows * _vocab(model) * hidden
    read += width * _vocab(model) * hidden + 4.0 * rows * _vocab(model)
    return flops, read


def work(case):
    kind = case["kind"]
    if kind == "request":
        parts = [_pass_work(case["model"], case["dtype"], 1, a, b - a, len(rows)) for a, b, rows in _portions(case)]
    elif kind == "batch":
        parts = [_pass_work(case["model"], "float32", case["batch"], 0, case["prompt"], case["batch"] * case["prompt"])]
        parts[0] = (parts[0][0], parts[0][1] - 4.0 * (case["batch"] * case["prompt"] - case["rows"]) * _vocab(case["model"]))
    elif kind == "generate":
        b, n = case["batch"], case["prompt"]
        parts = [_pass_work(case["model"], "float32", b, 0, n, b * n)] + [_pass_work(case["model"], "float32", b, n + i, 1, b) for i in range(case["decode"])]
    elif kind == "mlp":
        r, i, h, o = case["rows"], case["inputs"], case["hidden"], case["outputs"]
        parts = [(2.0 * r * (i * h + h * o), 4.0 * (r * i + i * h + h + h * o + o + r * o))]
    elif kind == "narrow":
        r, w, h, o = case["rows"], case["width"], case["hidden"], case["classes"]
        parts = [(2.0 * r * (3 * w * h + w * o), (1 if case["dtype"] == "float8" else 2) * (r * w + 3.0 * w * h + w * o) + 4.0 * r * o)]
    else:
        n = case["rows"] * case["cols"]
        parts = [(4.0 * n, (4 if case["dtype"] == "float32" else 2) * n + 8.0 * case["rows"])]
    return {"flops": float(sum(p[0] for p in parts)), "bytes": float(sum(p[1] for p in parts))}


# ------------------------------------------------------------------------------------------------ the same in 64 bits

def _wide(model, dtype):
    """name -> the weight in 64 bits, widened when it is asked for."""
    if (model, dtype) not in _weights:
        _weights.clear()
        torch.cuda.empty_cache()
        _weights[model, dtype] = {n: _weight(model, n, s, dtype) for n, s in _shapes(model)}
    w = _weights[model, dtype]
    return lambda name: w[name].double()


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _causal(n, window=None):
    i, j = torch.arange(n, device="cuda")[:, None], torch.arange(n, device="cuda")[None, :]
    return (j <= i) if window is None else (j <= i) & (i - j < window)


def _dense_hidden(model, W, ids):
    c, r = DENSE[model], DENSE[model].arch
    B, S = ids.shape
    h, g, hd, eps = c.num_attention_heads, c.num_key_value_heads, c.hd, c.rms_norm_eps
    x = W(f"{r}.model.embed_tokens.weight")[ids]
    angle = torch.arange(S, device="cuda").double()[:, None] * (1.0 / c.rope_theta ** (torch.arange(hd // 2, device="cuda").double() * 2.0 / hd))
    cos, sin = torch.cos(angle).repeat(1, 2), torch.sin(angle).repeat(1, 2)
    turn = lambda t: t * cos + torch.cat([-t[..., hd // 2:], t[..., : hd // 2]], -1) * sin  # noqa: E731
    hidden = ~_causal(S)
    for l in range(c.num_hidden_layers):
        p = f"{r}.model.layers.{l}"
        y = _rms(x, eps) * W(f"{p}.input_layernorm.weight")
        heads = lambda name, n: (y @ W(f"{p}.self_attn.{name}.weight").T).view(B, S, n, hd).transpose(1, 2)  # noqa: E731
        q, k, v = heads("q_proj", h), heads("k_proj", g), heads("v_proj", g)
        if r == "qwen3":
            q, k = _rms(q, eps) * W(f"{p}.self_attn.q_norm.weight"), _rms(k, eps) * W(f"{p}.self_attn.k_norm.weight")
        q, k = turn(q), turn(k)
        out = torch.empty_like(q)
        for b in range(B):
            for j in range(g):
                at = slice(j * (h // g), (j + 1) * (h // g))
                w = torch.softmax((q[b, at] @ k[b, j].T / math.sqrt(hd)).masked_fill(hidden, -math.inf), -1)
                out[b, at] = w @ v[b, j]
        x = x + out.transpose(1, 2).reshape(B, S, h * hd) @ W(f"{p}.self_attn.o_proj.weight").T
        y = _rms(x, eps) * W(f"{p}.post_attention_layernorm.weight")
        gate = y @ W(f"{p}.mlp.gate_proj.weight").T
        x = x + (gate * torch.sigmoid(gate) * (y @ W(f"{p}.mlp.up_proj.weight").T)) @ W(f"{p}.mlp.down_proj.weight").T
    return _rms(x, eps) * W(f"{r}.model.norm.weight"), W(f"{r}.model.embed_tokens.weight" if c.tie_word_embeddings else f"{r}.lm_head.weight")


def _runs(config):
    n, lp = len(config["layers"]), config["loop"]
    out = [(i, None) for i in range(lp["start"])]
    for t in range(lp["times"]):
        out += [(i, t if i == lp["start"] else None) for i in range(lp["start"], lp["stop"])]
    return out + [(i, None) for i in range(lp["stop"], n)]


def _taps(x, w):
    """Causal filter along the tokens, channel by channel: x [B, S, C], w [C, n] in time order."""
    n, S = w.shape[1], x.shape[1]
    p = torch.cat([torch.zeros_like(x[:, : n - 1]) if S >= n - 1 else x.new_zeros(x.shape[0], n - 1, x.shape[2]), x], 1)
    return sum(p[:, t:t + S] * w[:, t] for t in range(n))


def _loretar_attention(y, W, p, m, eps):
    B, S, _ = y.shape
    H, G, dk, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    pos = torch.arange(S, device="cuda").double()
    q = _rms(y @ W(p + ".q").T, eps) * W(p + ".q.norm")
    q = q * (1.0 + m["q_temp"]["coef"] * torch.log(torch.floor((pos + 1) / m["q_temp"]["every"]) + 1.0))[:, None]
    k = _rms(y @ W(p + ".k").T, eps) * W(p + ".k.norm")
    q, k, v = q.view(B, S, H, dk), k.view(B, S, G, dk), (y @ W(p + ".v").T).view(B, S, G, dv)
    slopes = 2.0 ** (-8.0 * (torch.arange(H, device="cuda").double() + 1) / H)
    seen, away, talk = _causal(S, m["mask"]["size"]), pos[:, None] - pos[None, :], W(p + ".talk")
    out = y.new_empty(B, S, H * dv)
    for b in range(B):
        s = torch.stack([q[b, :, h] @ k[b, :, h // (H // G)].T for h in range(H)]) * m["scale"] - slopes[:, None, None] * away
        w = torch.softmax(s.masked_fill_(~seen, -math.inf), -1)
        w = (talk @ w.view(H, S * S)).view(H, S, S)
        out[b] = torch.cat([w[h] @ v[b, :, h // (H // G)] for h in range(H)], -1)
    return out @ W(p + ".o").T


def _loretar_delta(y, W, p, m, eps):
    B, S, _ = y.shape
    H, G, dk, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    silu = torch.nn.functional.silu
    q = silu(_taps(y @ W(p + ".q").T, W(p + ".q.conv"))).view(B, S, G, dk)
    k = silu(_taps(y @ W(p + ".k").T, W(p + ".k.conv"))).view(B, S, G, dk)
    v = silu(_taps(y @ W(p + ".v").T, W(p + ".v.conv"))).view(B, S, H, dv)
    unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q, k = (unit(q) * dk ** -0.5).repeat_interleave(H // G, 2), unit(k).repeat_interleave(H // G, 2)
    beta = torch.sigmoid(y @ W(p + ".b").T)
    decay = torch.nn.functional.softplus((y @ W(p + ".a1").T) @ W(p + ".a2").T + W(p + ".dt_bias"), threshold=60.0).view(B, S, H, dk)
    decay = torch.exp(-torch.exp(W(p + ".A_log"))[:, None] * decay)
    st, o = y.new_zeros(B, H, dk, dv), torch.empty_like(v)
    for t in range(S):
        st = decay[:, t, :, :, None] * st
        u = beta[:, t, :, None] * (v[:, t] - (k[:, t, :, None] @ st)[:, :, 0])
        st = st + k[:, t, :, :, None] * u[:, :, None]
        o[:, t] = (q[:, t, :, None] @ st)[:, :, 0]
    gate = torch.sigmoid((y @ W(p + ".g1").T) @ W(p + ".g2").T).view(B, S, H, dv)
    return (_rms(o, eps) * W(p + ".norm") * gate).reshape(B, S, H * dv) @ W(p + ".o").T


def _loretar_hidden(model, W, ids):
    c, eps = BLOCKS[model], BLOCKS[model]["norm"]["eps"]
    x0 = x = W("embed")[ids]
    for i, begins in _runs(c):
        l, p = c["layers"][i], f"l{i}"
        if begins is not None:
            x = torch.cat([x, x0], -1) @ W("loop.in").T + W("loop.step")[begins]
        y = _rms(x, eps) * W(p + ".norm1")
        gate = lambda n: torch.sigmoid(y @ W(f"{p}.{n}").T + W(f"{p}.{n}.b"))  # noqa: E731
        mixed = (_loretar_attention if l["type"] == "attention" else _loretar_delta)(y, W, p + ".mix", l["mixer"], eps) * gate("rg1")
        z, a = y @ W(p + ".mlp.up").T, W(p + ".mlp.act")
        z = a[0] * _rms(z, eps) + a[1] * _rms(z ** 2, eps) + a[2] * _rms(z ** 3, eps) + a[3]
        x = x + mixed + (z @ W(p + ".mlp.down").T) * gate("rg2")
    return _rms(x, eps) * W("final.norm"), W("head")


def _group_norm(x, w, groups, eps):
    return _rms(x.view(x.shape[:-1] + (groups, -1)), eps).view(x.shape) * w


def _lufatar_attention(y, W, p, m, eps):
    B, S, _ = y.shape
    H, G, dk, dv, rot = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["rot"]["dims"]
    a = torch.arange(S, device="cuda").double()[:, None] * m["rot"]["base"] ** (-2.0 * torch.arange(rot // 2, device="cuda").double() / rot)
    co, si = torch.cos(a)[:, None], torch.sin(a)[:, None]

    def turn(t):
        u, v = t[..., 0:rot:2], t[..., 1:rot:2]
        return _rms(torch.cat([torch.stack([u * co - v * si, v * co + u * si], -1).flatten(-2), t[..., rot:]], -1), eps)

    q, k = turn((y @ W(p + ".q").T).view(B, S, H, dk)), turn((y @ W(p + ".k").T).view(B, S, G, dk))
    v, talk, seen = (y @ W(p + ".v").T).view(B, S, G, dv), W(p + ".talk"), _causal(S)
    out = y.new_empty(B, S, H * dv)
    for b in range(B):
        s = torch.stack([q[b, :, h] @ k[b, :, h // (H // G)].T for h in range(H)]) * m["scale"]
        s = (talk @ s.view(H, S * S)).view(H, S, S).masked_fill_(~seen, -math.inf)
        w = torch.softmax(torch.cat([s, s.new_zeros(H, S, 1)], -1), -1)[..., :S]
        out[b] = torch.cat([w[h] @ v[b, :, h // (H // G)] for h in range(H)], -1)
    return out @ W(p + ".o").T


def _lufatar_experts(y, W, p, f):
    shape, y, r = y.shape, y.reshape(-1, y.shape[-1]), f["router"]
    n, groups, limit = r["experts"], r["groups"], f["expert"]["limit"]
    s = torch.sigmoid(y @ W(p + ".router").T)
    choice = (s + W(p + ".correction")).view(-1, groups["count"], n // groups["count"])
    best = choice.topk(min(2, choice.shape[-1]), -1).values.sum(-1).topk(groups["keep"], -1).indices
    allowed = torch.full_like(choice, -math.inf).scatter_(1, best[..., None].expand(-1, -1, choice.shape[-1]), 0.0) + choice
    chosen = allowed.view(-1, n).topk(r["top"], -1).indices
    out = torch.zeros_like(y)
    for e in range(n):
        rows = (chosen == e).any(-1).nonzero()[:, 0]
        if rows.numel():
            h, q = y[rows], f"{p}.e{e}"
            g, u = (h @ W(q + ".gate").T).clamp(max=limit), (h @ W(q + ".up").T).clamp(-limit, limit)
            out[rows] += s[rows, e, None] * ((g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ W(q + ".down").T)
    return out.view(shape)


def _lufatar_hidden(model, W, ids):
    c = BLOCKS[model]
    eps, groups, mult, side, e = c["norm"]["eps"], c["norm"]["groups"], c["residual_mult"], c["token_side"]["dim"], c["embedding"]["bigram"]
    pair = torch.full_like(ids, e["buckets"])
    pair[:, 1:] = (ids[:, :-1] * e["mul_prev"] + ids[:, 1:] * e["mul_cur"]) % e["buckets"]
    x, own = W("embed")[ids] + W("bigram")[pair], W("side.embed")[ids]
    for i, begins in _runs(c):
        l, p = c["layers"][i], f"l{i}"
        if begins is not None:
            x = x + W("loop.step")[begins]
        normed = lambda n: _group_norm(x, W(f"{p}.norm{n}"), groups, eps)  # noqa: E731
        a, b = normed(1), normed(2)
        a, b = a + _taps(a, W(p + ".canon1")), b + _taps(b, W(p + ".canon2"))
        x = x + mult * (_lufatar_attention(a, W, p + ".mix", l["mixer"], eps) + _lufatar_experts(b, W, p + ".mlp", l["mlp"]))
        z = torch.nn.functional.gelu(x @ W(p + ".side.gate").T, approximate="tanh") * own[..., i * side:(i + 1) * side]
        x = x + mult * _rms(z @ W(p + ".side.proj").T, eps) * W(p + ".side.norm")
    return _group_norm(x, W("final.norm"), groups, eps), W("head")


def _hidden(model, dtype, ids):
    """(the rows that the vocabulary projection multiplies, that projection) for token ids [B, S]."""
    W, ids = _wide(model, dtype), torch.from_numpy(ids.astype(np.int64)).cuda()
    f = _dense_hidden if model in DENSE else _loretar_hidden if model.startswith("loretar") else _lufatar_hidden
    return f(model, W, ids)


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "request":
            x, head = _hidden(case["model"], case["dtype"], _tokens(case, seed)[None])
            return [x[0, [a + r for r in rows]] @ head.T for a, _, rows in _portions(case)]
        if kind == "batch":
            ids = _tokens(case, seed)
            x, head = _hidden(case["model"], "float32", ids)
            x = x.reshape(-1, x.shape[-1])
            best = torch.cat([(x[a:a + 1024] @ head.T).argmax(-1) for a in range(0, len(x), 1024)])
            return {"ids": best.view(ids.shape), "logits": x[torch.from_numpy(_wanted_rows(case, seed).astype(np.int64)).cuda()] @ head.T}
        if kind == "generate":
            ids, out = _tokens(case, seed), []
            x, head = _hidden(case["model"], "float32", ids)
            first = x @ head.T
            for i in range(case["decode"] + 1):
                if i:
                    x, head = _hidden(case["model"], "float32", ids)
                out.append((x[:, -1] @ head.T).argmax(-1).cpu().numpy().astype(np.uint32))
                ids = np.concatenate([ids, out[-1][:, None]], 1)
            return {"tokens": np.stack(out), "logits": first}
        t = {k: v.double() for k, v in _tensors(case, seed).items()}
        if kind == "mlp":
            y = torch.sigmoid(t["x"] @ t["mlp.l1.weight"].T + t["mlp.l1.bias"]) @ t["mlp.l2.weight"].T + t["mlp.l2.bias"]
            return y[None]
        if kind == "narrow":  # every operation's result is of the dtype: that is what these operations are
            most = 448.0 if case["dtype"] == "float8" else math.inf
            r = lambda v: v.clamp(-most, most).to(NARROW[case["dtype"]][1]).double()  # noqa: E731
            g, u = r(t["x"] @ t["gate"].T), r(t["x"] @ t["up"].T)
            a = r(r(g / r(1.0 + r(torch.exp(-g)))) * u)
            return r(r(a @ t["down"].T) @ t["head"].T)
        return {"lse": torch.logsumexp(t["x"], -1, keepdim=True), "argmax": None}


def tolerance(case):
    """About four times what the present path is off `exact` by, over the listed cases and some drawn ones."""
    kind = case["kind"]
    if kind in ("mlp", "statistics"):
        return {"rel": 1e-6}
    if kind == "narrow":
        return {"rel": {"float8": 1e-2, "bfloat16": 3e-3, "float16": 1e-3}[case["dtype"]], "max": 0.5}
    if case.get("dtype") == "bfloat16":
        return {"rel": 0.03, "max": 0.5}
    if kind == "generate":
        return {"rel": 1e-5, "differ": 0.01}
    return {"rel": 1e-4 if case["model"].startswith(("llama", "lufatar")) else 2e-5, "differ": 0.01}
