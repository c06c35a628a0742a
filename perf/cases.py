"""The work that programs give this framework, as cases to time and compare.

A case is one pass of one kind:

  norm       add_rms_norm over a few or many rows: the smallest calls.
  head       greedy_token, the vocabulary projection with its argmax.
  attention  norm_rope_cache and causal grouped_attention over a prompt's tokens.
  model      a whole model's decode step, with the logits of its token.
  decode     one token of one sequence through a slice of a model.
  batch      one token of each of several sequences through a slice.
  verify     the k + 1 rows of a speculative verify pass through a slice.
  prefill    a prompt through a slice.

A slice holds a ninth of a model's layers and of its vocabulary (every
projection at its full width, every layer with weights of its own), so that a
pass keeps the proportions of the whole model's. Model passes are captured in a
HIP graph by `prepare` and replayed by `run`, as DecodeState and prefill() do.
The sizes are the model shapes of hackthenorth_amd.model.SHAPES at the context
lengths, batches, prompts and draft widths of the benchmark and the tests.

Values: projections N(0, 0.02), those that write the residual stream smaller by
the square root of its number of additions, as models are initialised, and
embedding rows N(0, 0.5), so that the stream carries more than one layer adds,
as in a trained model; RMSNorm gains around 1, 8-bit weights as a symmetric
per-row quantisation of normal weights gives them, earlier K/V slots N(0, 1),
token ids uniform.
"""
import math

import torch

from hackthenorth_amd.decode import KVCache, RotaryTable, forward
from hackthenorth_amd.kernels.attention import grouped_attention
from hackthenorth_amd.kernels.fused import norm_rope_cache
from hackthenorth_amd.kernels.greedy import greedy_token
from hackthenorth_amd.kernels.projection import norm_projection
from hackthenorth_amd.kernels.rmsnorm import add_rms_norm
from hackthenorth_amd.model import SHAPES, Norm, Qwen3Model, shape_config
from hackthenorth_amd.quant import QuantizedWeight

DEVICE = "cuda"
EPS = 1e-6
THETA = 1e6
HEAD_DIM = 128
SLICE = 9        # a slice has 1 / SLICE of a model's layers and vocabulary
HEADROOM = 64    # cache slots after a pass's own: the request's later tokens
SLICES = ("decode", "batch", "verify", "prefill")


def listed():
    return [
        # One row's residual add and norm: what a launch costs.
        {"name": "norm_1row", "kind": "norm", "shape": "qwen3-0.6b", "rows": 1},
        # The vocabulary scores of a five-row verify pass.
        {"name": "head_8b_5rows", "kind": "head", "shape": "qwen3-8b", "rows": 5},
        # A whole small model's step: some 140 short dependent launches.
        {"name": "model_0.6b_step", "kind": "model", "shape": "qwen3-0.6b", "format": "bf16",
         "batch": 1, "tokens": 1, "context": 540},
        # Batch-one decode, the framework's first purpose.
        {"name": "decode_8b_bf16", "kind": "decode", "shape": "qwen3-8b", "format": "bf16",
         "batch": 1, "tokens": 1, "context": 2048},
        # The same with 8-bit weights at a long context.
        {"name": "decode_8b_int8", "kind": "decode", "shape": "qwen3-8b", "format": "int8",
         "batch": 1, "tokens": 1, "context": 8200},
        # A context at which the K/V cache counts as much as the weights.
        {"name": "decode_4b_fp8_long", "kind": "decode", "shape": "qwen3-4b",
         "format": "fp8_e4m3", "batch": 1, "tokens": 1, "context": 30011},
        # A server's batch of sequences.
        {"name": "batch_8b_16", "kind": "batch", "shape": "qwen3-8b", "format": "bf16",
         "batch": 16, "tokens": 1, "context": 512},
        # A draft model's four proposals and the current token.
        {"name": "verify_4b_5rows", "kind": "verify", "shape": "qwen3-4b", "format": "bf16",
         "batch": 1, "tokens": 5, "context": 4096},
        # A short prompt of odd length.
        {"name": "prefill_8b_201", "kind": "prefill", "shape": "qwen3-8b", "format": "bf16",
         "batch": 1, "tokens": 201, "context": 0},
        # A long prompt: the matrix cores' case.
        {"name": "prefill_8b_2048", "kind": "prefill", "shape": "qwen3-8b", "format": "bf16",
         "batch": 1, "tokens": 2048, "context": 0},
        # A prompt of a model with 8-bit weights.
        {"name": "prefill_4b_fp8_300", "kind": "prefill", "shape": "qwen3-4b",
         "format": "fp8_e4m3", "batch": 1, "tokens": 300, "context": 0},
        # A prompt longer than the captured ones: attention's share grows with its square.
        {"name": "attention_4b_5000", "kind": "attention", "shape": "qwen3-4b", "tokens": 5000,
         "context": 0},
    ]


def _log(rng, low, high):
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    shape = rng.choice(("qwen3-0.6b", "qwen3-4b", "qwen3-8b"))
    form = rng.choice(("bf16", "int8", "fp8_e4m3"))
    kind = rng.choice(("norm", "head", "attention", "model", "decode", "batch", "verify",
                       "prefill", "prefill"))
    if kind == "norm":
        return {"kind": kind, "shape": shape, "rows": _log(rng, 1, 4096)}
    if kind == "head":
        return {"kind": kind, "shape": shape, "rows": _log(rng, 1, 32)}
    if kind == "attention":
        return {"kind": kind, "shape": shape, "tokens": _log(rng, 33, 5000),
                "context": rng.choice((0, rng.randrange(1, 2000)))}
    case = {"kind": kind, "shape": shape, "format": form, "batch": 1, "tokens": 1,
            "context": 0}
    if kind == "model":
        case.update(shape="qwen3-0.6b", context=_log(rng, 32, 4096))
    elif kind == "decode":
        case["context"] = _log(rng, 64, 32000)
    elif kind == "batch":
        case.update(batch=_log(rng, 2, 32), context=_log(rng, 64, 4096))
    elif kind == "verify":
        case.update(tokens=_log(rng, 2, 16), context=_log(rng, 64, 8192))
    else:
        case["tokens"] = _log(rng, 16, 2048 if form == "bf16" else 300)
    return case


# ---------------------------------------------------------------- inputs


def _rng(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _normal(g, *shape, std=1.0):
    return torch.empty(shape, dtype=torch.bfloat16, device=DEVICE).normal_(0, std, generator=g)


def _gain(g, n):
    return (1 + 0.1 * torch.randn(n, generator=g, device=DEVICE)).to(torch.bfloat16)


def _weight(g, rows, cols, form, std=0.02):
    """A projection: bf16, or (codes, row scales)."""
    if form == "bf16":
        return _normal(g, rows, cols, std=std)
    # A quantised row's largest weight, some four deviations out, has the largest code.
    scale = torch.empty(rows, device=DEVICE).uniform_(0.8, 1.2, generator=g)
    if form == "int8":
        codes = _normal(g, rows, cols, std=30.0).round_().clamp_(-127, 127).to(torch.int8)
        return codes.view(torch.uint8), scale * (std / 30)
    codes = _normal(g, rows, cols, std=110.0).clamp_(-448, 448).to(torch.float8_e4m3fn)
    return codes.view(torch.uint8), scale * (std / 110)


def _config(case):
    s = SHAPES[case["shape"]]
    part = SLICE if case["kind"] in SLICES else 1
    return shape_config(case["shape"], num_hidden_layers=max(1, s["num_hidden_layers"] // part),
                        vocab_size=s["vocab_size"] // part,
                        weight_format=case.get("format", "bf16"))


def _model_inputs(case, seed):
    """Weights, ids, positions and earlier K/V of a model pass, as plain tensors."""
    c, g = _config(case), _rng(seed)
    form = c.weight_format
    b, t, ctx = case["batch"], case["tokens"], case["context"]
    adds = 0.02 / (2 * SHAPES[case["shape"]]["num_hidden_layers"]) ** 0.5
    layers = []
    for _ in range(c.num_hidden_layers):
        layers.append({
            "qkv": _weight(g, sum(c.widths), c.hidden_size, form),
            "o": _weight(g, c.hidden_size, c.widths[0], form, adds),
            "gate_up": _weight(g, 2 * c.intermediate_size, c.hidden_size, form),
            "down": _weight(g, c.hidden_size, c.intermediate_size, form, adds),
            "ln1": _gain(g, c.hidden_size), "ln2": _gain(g, c.hidden_size),
            "q_norm": _gain(g, c.head_dim), "k_norm": _gain(g, c.head_dim)})
    embed = _normal(g, c.vocab_size, c.hidden_size, std=0.5)
    tied = c.tie_word_embeddings and form == "bf16"
    return c, {
        "layers": layers, "embed": embed, "norm": _gain(g, c.hidden_size),
        "head": embed if tied else _weight(g, c.vocab_size, c.hidden_size, form),
        "ids": torch.randint(c.vocab_size, (b, t), generator=g, device=DEVICE),
        "positions": ctx + torch.arange(t, device=DEVICE),
        "past": _normal(g, c.num_hidden_layers, 2, b, c.num_key_value_heads, ctx, c.head_dim)}


def _held(w, form):
    return w if form == "bf16" else QuantizedWeight(w[0], w[1], form)


def _model(c, data):
    model = Qwen3Model(c, DEVICE)
    model.embed_weight = data["embed"]
    model.lm_head_weight = _held(data["head"], c.weight_format)
    model.norm = Norm(data["norm"], EPS)
    for layer, d in zip(model.layers, data["layers"]):
        for kind in ("qkv", "o", "gate_up", "down"):
            setattr(layer, kind + "_weight", _held(d[kind], c.weight_format))
        layer.input_layernorm = Norm(d["ln1"], EPS)
        layer.post_attention_layernorm = Norm(d["ln2"], EPS)
        layer.q_norm, layer.k_norm = Norm(d["q_norm"], EPS), Norm(d["k_norm"], EPS)
    return model


def _prepare_model(case, seed):
    c, data = _model_inputs(case, seed)
    model = _model(c, data)
    t, ctx = case["tokens"], case["context"]
    cache = KVCache(model, case["batch"], ctx + t + HEADROOM)
    cache.storage[..., :ctx, :] = data["past"]
    rotary = RotaryTable(model, cache.capacity)

    def step():
        hidden = []
        tokens = forward(model, data["ids"], cache, data["positions"], rotary=rotary,
                         last_only=case["kind"] != "verify", record=hidden)
        out = {"hidden": hidden[-1]}
        if case["kind"] == "model":
            out["logits"] = norm_projection(hidden[-1], model.norm.weight,
                                            model.lm_head_weight, EPS)
        return tokens, out

    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.inference_mode(), torch.cuda.stream(stream):
        step()  # library load and workspaces, outside of the capture
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.inference_mode(), torch.cuda.graph(graph, stream=stream):
        tokens, out = step()
    out["appended"] = cache.storage[..., ctx:ctx + t, :]
    return {"kind": case["kind"], "graph": graph, "out": out,
            "kept": (model, cache, rotary, data, tokens)}


def _norm_inputs(case, seed):
    g, cols = _rng(seed), SHAPES[case["shape"]]["hidden_size"]
    return {"x": _normal(g, case["rows"], cols, std=0.5),
            "residual": _normal(g, case["rows"], cols), "gain": _gain(g, cols)}


def _head_inputs(case, seed):
    """Hidden rows of a model that is sure of its next token, as a trained one mostly is."""
    g, s = _rng(seed), SHAPES[case["shape"]]
    k, rows = s["hidden_size"], case["rows"]
    weight = _normal(g, s["vocab_size"], k, std=0.02)
    ids = torch.randint(s["vocab_size"], (rows,), generator=g, device=DEVICE)
    own = weight[ids].float()
    own = own * (0.25 * k ** 0.5 / own.norm(dim=-1, keepdim=True))
    return {"x": (torch.randn(rows, k, generator=g, device=DEVICE) + own).to(torch.bfloat16),
            "weight": weight}


def _attention_inputs(case, seed):
    g, s = _rng(seed), SHAPES[case["shape"]]
    hq, hkv = s["num_attention_heads"], s["num_key_value_heads"]
    t, ctx = case["tokens"], case["context"]
    angles = _angles(ctx + torch.arange(t, device=DEVICE))
    return {"packed": _normal(g, 1, t, hq + 2 * hkv, HEAD_DIM),
            "cos": angles.cos().to(torch.bfloat16)[None],
            "sin": angles.sin().to(torch.bfloat16)[None],
            "q_norm": _gain(g, HEAD_DIM), "k_norm": _gain(g, HEAD_DIM),
            "positions": ctx + torch.arange(t, device=DEVICE),
            "past": _normal(g, 2, 1, hkv, ctx, HEAD_DIM)}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "norm":
        return {"kind": kind, **_norm_inputs(case, seed)}
    if kind == "head":
        return {"kind": kind, **_head_inputs(case, seed)}
    if kind == "attention":
        d = _attention_inputs(case, seed)
        s, t, ctx = SHAPES[case["shape"]], case["tokens"], case["context"]
        hq, hkv = s["num_attention_heads"], s["num_key_value_heads"]
        cache = torch.zeros((2, 1, hkv, ctx + t + HEADROOM, HEAD_DIM), dtype=torch.bfloat16,
                            device=DEVICE)
        cache[..., :ctx, :] = d["past"]
        q, k, v = d["packed"].split((hq, hkv, hkv), 2)
        return {"kind": kind, "q": q, "k": k, "v": v, "cache": cache,
                "norms": (Norm(d["q_norm"], EPS), Norm(d["k_norm"], EPS)),
                "appended": cache[..., ctx:ctx + t, :], **d}
    return _prepare_model(case, seed)


def run(state):
    kind = state["kind"]
    if kind == "norm":
        return add_rms_norm(state["x"], state["residual"], state["gain"], EPS)
    if kind == "head":
        return greedy_token(state["x"], state["weight"])
    if kind == "attention":
        keys, values = state["cache"]
        q, _, _ = norm_rope_cache(state["q"], state["k"], state["v"], *state["norms"],
                                  state["cos"], state["sin"], keys, values, state["positions"])
        return {"out": grouped_attention(q, keys, values, state["positions"]),
                "appended": state["appended"]}
    state["graph"].replay()
    return state["out"]


# ---------------------------------------------------------------- what a pass cannot do without


def _visible(tokens, context):
    """Cache slots that the tokens' queries see, summed over the queries."""
    return tokens * context + tokens * (tokens + 1) // 2


def work(case):
    kind, s = case["kind"], SHAPES[case["shape"]]
    h, hq, hkv = s["hidden_size"], s["num_attention_heads"], s["num_key_value_heads"]
    if kind == "norm":
        return {"bytes": 2 * h * (4 * case["rows"] + 1), "flops": 5 * h * case["rows"]}
    if kind == "head":
        return {"bytes": 2 * h * (s["vocab_size"] + case["rows"]) + 8 * case["rows"],
                "flops": 2 * case["rows"] * h * s["vocab_size"]}
    t, ctx = case["tokens"], case["context"]
    if kind == "attention":
        heads = (hq + 2 * hkv) + hq + 2 * hkv  # packed in; rows and cache slots out
        return {"bytes": 2 * HEAD_DIM * (t * heads + 2 * t + 2 * hkv * ctx),
                "flops": 4 * HEAD_DIM * hq * _visible(t, ctx)}
    c, b = _config(case), case["batch"]
    wide = 1 if c.quantized else 2
    weights = (sum(c.widths) + c.widths[0] + 3 * c.intermediate_size) * h
    scored = b * (t if kind == "verify" else 1)
    kv = 2 * 2 * hkv * HEAD_DIM
    layers = c.num_hidden_layers
    return {"bytes": wide * (layers * weights + c.vocab_size * h)
            + layers * b * (ctx + 2 * t) * kv + 4 * h * b * t,
            "flops": 2 * b * t * layers * weights + 2 * scored * c.vocab_size * h
            + layers * b * 4 * HEAD_DIM * hq * _visible(t, ctx)}


def tolerance(case):
    kind = case["kind"]
    if kind == "head":
        return "exact"
    if kind == "norm":
        # Two roundings to bf16 of values that 32-bit sums may move across a boundary.
        return {"rel": 2e-3, "max": 2e-2}
    if kind == "attention":
        # 32-bit sums in another order, rounded to bf16 once.
        return {"rel": 4e-3, "max": 4e-2}
    # bf16 rows between the operations: one value rounded the other way in one
    # layer moves every value of the layers after it. The one-row kernels and
    # the multi-row ones, which sum in other orders, are 2e-3 to 7e-3 apart on
    # these slices (largest single difference 0.042) and up to 8e-3 on the
    # whole model.
    return {"rel": 2.5e-2 if kind != "model" else 3e-2, "max": 2e-1}


# ---------------------------------------------------------------- the same in 64 bits


def _wide(w, form):
    if form == "bf16":
        return w.double()
    codes, scale = w
    codes = codes.view(torch.int8 if form == "int8" else torch.float8_e4m3fn)
    return codes.float().double() * scale.double()[:, None]


def _angles(positions):
    inv = 1.0 / THETA ** (torch.arange(0, HEAD_DIM, 2, device=DEVICE).double() / HEAD_DIM)
    a = positions.double()[:, None] * inv[None, :]
    return torch.cat((a, a), dim=-1)


def _rms(x, gain):
    return gain.double() * x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def _rope(x, angles):
    """x [B, T, heads, 128] turned by the tokens' angles [T, 128]."""
    half = torch.cat((-x[..., HEAD_DIM // 2:], x[..., :HEAD_DIM // 2]), dim=-1)
    return x * angles.cos()[None, :, None] + half * angles.sin()[None, :, None]


def _attend(q, keys, values, positions):
    """q [B, T, Hq, 128] over caches [B, Hkv, S, 128]; returns q's shape."""
    b, _, hq, _ = q.shape
    group = hq // keys.shape[1]
    hidden = torch.arange(keys.shape[2], device=DEVICE)[None, :] > positions[:, None]
    out = torch.empty_like(q)
    for i in range(b):
        for h in range(hq):
            scores = q[i, :, h] @ keys[i, h // group].T / HEAD_DIM ** 0.5
            weights = scores.masked_fill_(hidden, -math.inf).softmax(-1)
            out[i, :, h] = weights @ values[i, h // group]
    return out


def _exact_model(case, seed):
    c, data = _model_inputs(case, seed)
    b, t = data["ids"].shape
    hq, hkv = c.num_attention_heads, c.num_key_value_heads
    angles = _angles(data["positions"])
    h = data["embed"][data["ids"]].double()
    form, appended = c.weight_format, []
    for d, past in zip(data["layers"], data["past"]):
        x = _rms(h, d["ln1"]) @ _wide(d["qkv"], form).T
        q, k, v = x.view(b, t, hq + 2 * hkv, HEAD_DIM).split((hq, hkv, hkv), 2)
        q, k = _rope(_rms(q, d["q_norm"]), angles), _rope(_rms(k, d["k_norm"]), angles)
        new = torch.stack((k, v)).transpose(2, 3)
        appended.append(new)
        keys, values = torch.cat((past.double(), new), dim=3)
        a = _attend(q, keys, values, data["positions"]).reshape(b, t, -1)
        h = h + a @ _wide(d["o"], form).T
        gate, up = (_rms(h, d["ln2"]) @ _wide(d["gate_up"], form).T).chunk(2, dim=-1)
        h = h + (torch.nn.functional.silu(gate) * up) @ _wide(d["down"], form).T
    out = {"hidden": h, "appended": torch.stack(appended)}
    if case["kind"] == "model":
        out["logits"] = _rms(h, data["norm"]) @ _wide(data["head"], form).T
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "norm":
        d = _norm_inputs(case, seed)
        total = d["x"].double() + d["residual"].double()
        return total, _rms(total, d["gain"])
    if kind == "head":
        d = _head_inputs(case, seed)
        best = []
        for part in d["weight"].split(1 << 14):
            best.append((d["x"].double() @ part.double().T).max(dim=-1))
        top = torch.stack([p.values for p in best]).argmax(dim=0)
        at = torch.stack([p.indices for p in best])
        return top * (1 << 14) + at.gather(0, top[None])[0]
    if kind == "attention":
        d = _attention_inputs(case, seed)
        s = SHAPES[case["shape"]]
        hq, hkv = s["num_attention_heads"], s["num_key_value_heads"]
        q, k, v = d["packed"].double().split((hq, hkv, hkv), 2)
        angles = _angles(d["positions"])
        q, k = _rope(_rms(q, d["q_norm"]), angles), _rope(_rms(k, d["k_norm"]), angles)
        new = torch.stack((k, v)).transpose(2, 3)
        keys, values = torch.cat((d["past"].double(), new), dim=3)
        return {"out": _attend(q, keys, values, d["positions"]).transpose(1, 2),
                "appended": new}
    return _exact_model(case, seed)
