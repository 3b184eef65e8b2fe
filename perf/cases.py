"""The calls whose speed is tracked, as a user's program makes them.

Six kinds of call, each through a public entry point, over the shapes of the 3B- and 27B-class
decoders of ``texelator_amd.modeling`` and generic odd sizes:

* ``linear``            ``runtime.TexelatorLinear`` on one BC4 handle: decode (one token), batched decode
                        (a few sequences or drafted tokens, below the prefill threshold), prompts of
                        any length; bf16 or fp16; with or without the handle's bias; the defined
                        palette or an artifact's own palette table.
* ``decode_attention``  one query token over a KV cache (``layers.decode_attention``).
* ``prompt_attention``  the causal attention of a prompt (``layers.prefill_attention``).
* ``decode_step``       one token through a whole ``BC4Decoder`` to its logits, captured once as a graph
                        and replayed, as ``BC4Decoder.decode`` runs it.
* ``prefill``           a prompt through a ``BC4Decoder`` to its hidden states and last logits.
* ``encode``            a dense matrix to BC4 blocks on the GPU (``encoder.encode_matrix_tensor``), as a
                        conversion runs it per linear.
"""
from __future__ import annotations

import math
import weakref

import torch

from texelator_amd import encoder, layers, runtime
from texelator_amd.modeling import BC4Decoder, DecoderConfig

HEAD_DIM = 128
# (hidden, heads, kv_heads, intermediate) of the two decoder classes
CLASSES = {"3b": (2048, 16, 2, 11008), "27b": (5120, 40, 8, 27648)}
VOCAB = 32768
MAX_WEIGHTS = 27648 * 5120
MAX_TOKENS = 2048


def _linear(name: str, m: int, k: int, tokens: int, dtype: str = "bf16", bias: bool = False, lut: bool = False) -> dict:
    return {"name": name, "kind": "linear", "m": m, "k": k, "tokens": tokens, "dtype": dtype, "bias": bias, "lut": lut}


def listed() -> list[dict]:
    return [
        # one decoded token through the smallest linear: k or v projection, 3B class, with its bias
        _linear("decode_kv_3b", 256, 2048, 1, bias=True),
        # one decoded token through the largest linear: gate or up projection, 27B class
        _linear("decode_gate_27b", 27648, 5120, 1),
        # eight sequences decoded together (or eight drafted tokens checked): down projection
        _linear("batch8_down_27b", 5120, 27648, 8),
        # a short chat prompt of ragged length: q or o projection
        _linear("prompt77_q_27b", 5120, 5120, 77),
        # a long prompt: gate or up projection
        _linear("prompt2048_gate_27b", 27648, 5120, 2048),
        # fp16 activations (artifacts with runtime_dtype float16), no size a multiple of a tile
        _linear("prompt333_fp16_odd", 3000, 4848, 333, dtype="fp16", bias=True),
        # an artifact encoded against another GPU's palette, which it brings as a table: decode
        _linear("decode_lut_17408", 17408, 5120, 1, lut=True),
        # attention of one decoded token in a 4096-token conversation, 27B class
        {"name": "decode_attention_4k", "kind": "decode_attention", "heads": 40, "kv_heads": 8, "position": 4000,
         "length": 4096},
        # attention of a prompt of about a thousand tokens, 27B class
        {"name": "prompt_attention_1000", "kind": "prompt_attention", "heads": 40, "kv_heads": 8, "tokens": 1000},
        # a decoded token through a 3B-class decoder, 700 tokens into its conversation
        {"name": "decode_step_3b", "kind": "decode_step", "class": "3b", "layers": 8, "position": 700},
        # a 512-token prompt through a 27B-class layer
        {"name": "prefill512_27b", "kind": "prefill", "class": "27b", "layers": 1, "tokens": 512},
        # conversion of a 27B-class q or o projection
        {"name": "encode_5120", "kind": "encode", "m": 5120, "k": 5120, "dtype": "bf16"},
    ]


def _spread(rng, low: float, high: float) -> int:
    """An integer spread evenly over the logarithm of [low, high]."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng) -> dict:
    kind = rng.choices(["linear", "decode_attention", "prompt_attention", "decode_step", "prefill", "encode"],
                       [8, 1, 1, 1, 1, 1])[0]
    if kind == "linear":
        k = 16 * _spread(rng, 128, 1728)
        m = _spread(rng, 256, min(27648, MAX_WEIGHTS // k))
        tokens = rng.choice([1, 1, rng.randint(2, 15), _spread(rng, 16, MAX_TOKENS), _spread(rng, 16, MAX_TOKENS)])
        return {"kind": kind, "m": m, "k": k, "tokens": tokens, "dtype": rng.choice(["bf16", "bf16", "bf16", "fp16"]),
                "bias": rng.random() < 0.5, "lut": rng.random() < 0.15}
    if kind == "decode_attention":
        group, kv_heads = rng.choice([(1, 8), (2, 8), (5, 8), (8, 2), (7, 4), (4, 8)])
        length = 512 * _spread(rng, 1, 32)
        return {"kind": kind, "heads": group * kv_heads, "kv_heads": kv_heads, "position": rng.randrange(length),
                "length": length}
    if kind == "prompt_attention":
        heads, kv_heads = rng.choice([(40, 8), (16, 2), (32, 8), (28, 4)])
        return {"kind": kind, "heads": heads, "kv_heads": kv_heads, "tokens": _spread(rng, 16, 4096)}
    if kind == "decode_step":
        size = rng.choice(["3b", "27b"])
        return {"kind": kind, "class": size, "layers": rng.randint(1, 8 if size == "3b" else 2),
                "position": _spread(rng, 1, 4090)}
    if kind == "prefill":
        size = rng.choice(["3b", "27b"])
        return {"kind": kind, "class": size, "layers": rng.randint(1, 3) if size == "3b" else 1,
                "tokens": _spread(rng, 17, 600)}
    return {"kind": "encode", "m": _spread(rng, 256, 5120), "k": 16 * _spread(rng, 64, 320),
            "dtype": rng.choice(["bf16", "fp32"])}


# ---------------------------------------------------------------------------------------------
# Inputs (from the seed alone)


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g: torch.Generator, *shape: int, std: float = 1.0) -> torch.Tensor:
    return torch.randn(shape, device="cuda", generator=g) * std


def _palette() -> torch.Tensor:
    """The defined palette [255, 255, 8] (index e1 + 127, e0 + 127, selector) in float32: endpoints
    e / 127, six further steps of (e1 - e0) / 889 where e0 > e1, else four of (e1 - e0) / 635 and -1, 1;
    quotients and interpolants each rounded to float32 once."""
    e = torch.arange(-127, 128, device="cuda", dtype=torch.float64)
    e1, e0 = e[:, None], e[None, :]
    eight = e0 > e1
    rounded = lambda t: t.to(torch.float32).to(torch.float64)  # noqa: E731
    base, end = rounded(e0 / 127).expand(255, 255), rounded(e1 / 127).expand(255, 255)
    step = rounded(torch.where(eight, (e1 - e0) / 889, (e1 - e0) / 635))
    values = [base, end] + [base + s * step for s in range(1, 7)]
    values[6] = torch.where(eight, values[6], torch.full_like(base, -1.0))
    values[7] = torch.where(eight, values[7], torch.full_like(base, 1.0))
    return torch.stack(values, dim=-1).to(torch.float32)


def _foreign_palette() -> torch.Tensor:
    """Another GPU's palette: the defined one's interpolants in steps of 2^-14, as a sampler with
    fixed-point weights returns them; the endpoints as they are."""
    table = _palette()
    table[..., 2:] = torch.round(table[..., 2:] * 16384) / 16384
    return table.contiguous()


def _blocks(m: int, k: int, g: torch.Generator, std: float = 0.02) -> tuple[torch.Tensor, torch.Tensor]:
    """A normal matrix in BC4: row scale max |w|, a block's endpoints its largest and smallest
    value, selectors the nearest of the eight evenly spaced values. ``(blocks, scales)`` on the GPU."""
    blocks = torch.empty((m, k // 16), dtype=torch.int64, device="cuda")
    scales = torch.empty(m, dtype=torch.float32, device="cuda")
    shifts = 3 * torch.arange(16, device="cuda") + 16
    for first in range(0, m, 8192):
        rows = _normal(g, min(8192, m - first), k, std=std)
        scale = rows.abs().amax(1)
        values = (rows / scale[:, None]).view(rows.shape[0], -1, 16)
        e0, e1 = torch.round(values.amax(2) * 127), torch.round(values.amin(2) * 127)
        level = torch.round((e0[..., None] - values * 127) * (7 / (e0 - e1).clamp_min(1))[..., None]).clamp(0, 7).long()
        selector = torch.where(level == 0, level, torch.where(level == 7, torch.ones_like(level), level + 1))
        word = (selector << shifts).sum(2)
        blocks[first:first + rows.shape[0]] = word | (e0.long() & 0xFF) | ((e1.long() & 0xFF) << 8)
        scales[first:first + rows.shape[0]] = scale
    return blocks.view(torch.uint8).reshape(-1), scales


def _dense(blocks: torch.Tensor, scales: torch.Tensor, palette: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    """The weights the blocks stand for, [M, K] float64: palette value times row scale in float32,
    rounded to the activations' type."""
    m = scales.numel()
    raw = blocks.view(m, -1, 8)
    end = raw[..., :2].view(torch.int8).clamp_min(-127).long() + 127
    word = blocks.view(torch.int64).view(m, -1)
    table = palette.reshape(-1)
    row = (end[..., 1] * 255 + end[..., 0]) * 8
    out = torch.empty((m, raw.shape[1], 16), dtype=torch.float64, device="cuda")
    for position in range(16):
        selector = (word >> (16 + 3 * position)) & 7
        out[..., position] = (table[row + selector] * scales[:, None]).to(dtype).double()
    return out.view(m, -1)


def _activations(g: torch.Generator, tokens: int, k: int, dtype: torch.dtype) -> torch.Tensor:
    """Normalised hidden states: unit variance, channels of unequal size."""
    return (_normal(g, tokens, k) * torch.exp(0.3 * _normal(g, 1, k))).to(dtype)


def _dtype(case: dict) -> torch.dtype:
    return {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}[case["dtype"]]


def _linear_inputs(case: dict, seed: int) -> dict:
    g, dtype = _generator(seed), _dtype(case)
    blocks, scales = _blocks(case["m"], case["k"], g)
    return {"blocks": blocks, "scales": scales, "x": _activations(g, case["tokens"], case["k"], dtype),
            "bias": _normal(g, case["m"], std=0.5).to(dtype) if case["bias"] else None,
            "palette": _foreign_palette() if case["lut"] else None}


def _attention_inputs(case: dict, seed: int) -> dict:
    g = _generator(seed)
    heads, kv_heads = case["heads"], case["kv_heads"]
    tokens, length = (1, case["length"]) if case["kind"] == "decode_attention" else (case["tokens"], case["tokens"])
    bf16 = torch.bfloat16
    return {"q": _normal(g, tokens, heads * HEAD_DIM).to(bf16), "k": _normal(g, kv_heads, length, HEAD_DIM).to(bf16),
            "v": _normal(g, kv_heads, length, HEAD_DIM).to(bf16)}


def _encode_inputs(case: dict, seed: int) -> dict:
    g = _generator(seed)
    weight = (_normal(g, case["m"], case["k"], std=0.02) * torch.exp(0.3 * _normal(g, 1, case["k"]))).to(_dtype(case))
    return {"weight": weight, "moments": torch.exp(0.6 * _normal(g, case["k"])), "palette": _palette()}


def _config(case: dict) -> DecoderConfig:
    hidden, heads, kv_heads, intermediate = CLASSES[case["class"]]
    return DecoderConfig(layers=case["layers"], hidden=hidden, heads=heads, kv_heads=kv_heads, head_dim=HEAD_DIM,
                         intermediate=intermediate, vocab=VOCAB)


def _shapes(case: dict) -> dict[str, tuple[int, int]]:
    hidden, heads, kv_heads, inter = CLASSES[case["class"]]
    q, kv = heads * HEAD_DIM, kv_heads * HEAD_DIM
    return {"self_attn.q_proj": (q, hidden), "self_attn.k_proj": (kv, hidden), "self_attn.v_proj": (kv, hidden),
            "self_attn.o_proj": (hidden, q), "mlp.gate_proj": (inter, hidden), "mlp.up_proj": (inter, hidden),
            "mlp.down_proj": (hidden, inter)}


def _cached(case: dict) -> int:
    """Positions the model's cache holds."""
    return 4096 if case["kind"] == "decode_step" else case["tokens"]


def _model_inputs(case: dict, seed: int) -> dict:
    g, bf16 = _generator(seed), torch.bfloat16
    hidden, _, kv_heads, _ = CLASSES[case["class"]]
    weights = {}
    for name, (m, k) in _shapes(case).items():
        narrow = name.endswith(("o_proj", "down_proj"))  # residual projections: GPT-2's depth scaling
        weights[name] = _blocks(m, k, g, std=0.02 / math.sqrt(2 * case["layers"]) if narrow else 0.02)
    past = (case["layers"], kv_heads, _cached(case), HEAD_DIM)
    decode = case["kind"] == "decode_step"
    return {"weights": weights, "embed": _normal(g, VOCAB, hidden).to(bf16),
            "lm_head": _normal(g, VOCAB, hidden, std=0.02).to(bf16),
            "norms": [torch.exp(0.2 * _normal(g, hidden)).to(bf16) for _ in range(2 * case["layers"] + 1)],
            "ids": torch.randint(0, VOCAB, (1 if decode else case["tokens"],), device="cuda", generator=g),
            "k": _normal(g, *past).to(bf16) if decode else None, "v": _normal(g, *past).to(bf16) if decode else None}


# ---------------------------------------------------------------------------------------------
# What a program holds, and the call


class _Linear:
    """One packed matrix as a module; the handle goes with it."""

    def __init__(self, inputs: dict):
        ext = runtime.extension()
        handle = ext.pack_encoded_device(inputs["blocks"], inputs["scales"], inputs["bias"])
        if inputs["palette"] is not None:
            ext.set_palette_table(handle, inputs["palette"])
        self.module = runtime.TexelatorLinear([handle])
        weakref.finalize(self, ext.free, handle)


def _decoder(case: dict, inputs: dict) -> BC4Decoder:
    """A decoder of the case's class over the inputs' weights (every layer its own copy of them)."""
    model = BC4Decoder(_config(case), max_context=_cached(case),
                       linear_source=lambda layer, name, m, k: inputs["weights"][name])
    weakref.finalize(model, lambda handles: [runtime.extension().free(h) for h in handles], list(model.handles))
    model.embed, model.lm_head, model.final_norm = inputs["embed"], inputs["lm_head"], inputs["norms"][-1]
    for index, layer in enumerate(model.layers):
        layer.input_norm, layer.post_norm = inputs["norms"][2 * index:2 * index + 2]
    if inputs["k"] is not None:
        model.k_cache.copy_(inputs["k"])
        model.v_cache.copy_(inputs["v"])
    return model


@torch.inference_mode()
def _decode_graph(case: dict, inputs: dict) -> dict:
    model = _decoder(case, inputs)
    position = case["position"]
    length = min(model.max_context, (position // 512 + 1) * 512)
    model.token.copy_(inputs["ids"])
    model.position.fill_(position)
    logits = torch.empty(VOCAB, dtype=torch.bfloat16, device="cuda")
    token = torch.empty(1, dtype=torch.int64, device="cuda")

    def step():
        hidden = model.hidden_states(model.token, model.position, length)
        layers.lm_head_argmax(model.lm_head, hidden, model.head_workspace, out=token, logits=logits)

    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        step()
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        step()
    return {"model": model, "graph": graph, "logits": logits, "token": token}


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    state = {"kind": kind}
    if kind == "linear":
        inputs = _linear_inputs(case, seed)
        state.update(linear=_Linear(inputs), x=inputs["x"])
    elif kind == "decode_attention":
        state.update(_attention_inputs(case, seed), heads=case["heads"], kv_heads=case["kv_heads"], length=case["length"],
                     position=torch.tensor([case["position"]], device="cuda"))
        need = layers.decode_attention_workspace_bytes(case["heads"], case["length"])
        state["workspace"] = torch.empty(need, dtype=torch.uint8, device="cuda")
    elif kind == "prompt_attention":
        state.update(_attention_inputs(case, seed), heads=case["heads"], kv_heads=case["kv_heads"])
    elif kind == "decode_step":
        state.update(_decode_graph(case, _model_inputs(case, seed)))
    elif kind == "prefill":
        inputs = _model_inputs(case, seed)
        state.update(model=_decoder(case, inputs), ids=inputs["ids"])
    else:
        state.update(_encode_inputs(case, seed))
    return state


@torch.inference_mode()
def run(state: dict):
    kind = state["kind"]
    if kind == "linear":
        return state["linear"].module(state["x"])
    if kind == "decode_attention":
        return layers.decode_attention(state["q"], state["k"], state["v"], state["position"], state["length"],
                                       state["heads"], state["kv_heads"], 1 / math.sqrt(HEAD_DIM), state["workspace"])
    if kind == "prompt_attention":
        return layers.prefill_attention(state["q"], state["k"], state["v"], state["heads"], state["kv_heads"],
                                        1 / math.sqrt(HEAD_DIM))
    if kind == "decode_step":
        state["graph"].replay()
        return {"logits": state["logits"], "k": state["model"].k_cache, "v": state["model"].v_cache}
    if kind == "prefill":
        model, ids = state["model"], state["ids"]
        hidden = model.hidden_states(ids, model.key_positions[:ids.numel()], ids.numel())
        return {"hidden": hidden, "logits": model.logits(hidden[-1:]), "k": model.k_cache, "v": model.v_cache}
    blocks, scales = encoder.encode_matrix_tensor(state["weight"], state["moments"], state["palette"])
    return {"blocks": blocks, "scales": scales}


# ---------------------------------------------------------------------------------------------
# What a pass cannot do without


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "linear":
        m, k, t = case["m"], case["k"], case["tokens"]
        read = m * k // 2 + 4 * m + 2 * t * k + (2 * m if case["bias"] else 0) + (255 * 255 * 32 if case["lut"] else 0)
        return {"bytes": read + 2 * t * m, "flops": 2 * t * m * k}
    if kind == "decode_attention":
        keys = case["position"] + 1
        return {"bytes": 4 * HEAD_DIM * (keys * case["kv_heads"] + case["heads"]), "flops": 4 * HEAD_DIM * keys * case["heads"]}
    if kind == "prompt_attention":
        t = case["tokens"]
        return {"bytes": 4 * HEAD_DIM * t * (case["kv_heads"] + case["heads"]),
                "flops": 2 * HEAD_DIM * t * (t + 1) * case["heads"]}
    if kind == "encode":
        weights = case["m"] * case["k"]
        # a distance and a comparison per weight, palette value and searched palette (ten of them)
        return {"bytes": weights * (4 if case["dtype"] == "fp32" else 2) + weights // 2 + 4 * case["m"] + 4 * case["k"],
                "flops": 160 * weights}
    hidden, heads, kv_heads, _ = CLASSES[case["class"]]
    weights = case["layers"] * sum(m * k for m, k in _shapes(case).values())
    t = 1 if kind == "decode_step" else case["tokens"]
    keys = case["position"] + 1 if kind == "decode_step" else (t + 1) / 2
    past = case["layers"] * kv_heads * (keys if kind == "decode_step" else t) * HEAD_DIM * 4
    return {"bytes": int(weights // 2 + 2 * VOCAB * hidden + past + 2 * t * hidden),
            "flops": int(2 * t * weights + 2 * VOCAB * hidden + 4 * case["layers"] * t * keys * heads * HEAD_DIM)}


def tolerance(case: dict):
    if case["kind"] == "encode":
        # scales are exact maxima; endpoints tie where a sum of sixteen terms is taken in another order
        return {"rel": 1e-6, "differ": 1e-3}
    if case["kind"] in ("decode_step", "prefill"):
        # measured against 64 bits: 4e-3 (decode step), 8e-3 (prefill: bf16 activations into four linears a layer)
        return {"rel": 2e-2 if case["kind"] == "decode_step" else 3e-2, "max": 0.2}
    if case.get("dtype") == "fp16":
        return {"rel": 1.2e-3, "max": 1e-2}  # measured 2.9e-4: the output's rounding
    return {"rel": 8e-3, "max": 5e-2}  # measured 1.7e-3 (linears), 2.0e-3 (attention): the output's rounding


# ---------------------------------------------------------------------------------------------
# The same results in 64 bits


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, first: int) -> torch.Tensor:
    """q [T, heads, d] at positions first.. over keys and values [kv_heads, L, d], all float64."""
    tokens, heads, d = q.shape
    group = heads // k.shape[0]
    out = torch.empty_like(q)
    future = torch.arange(k.shape[1], device="cuda")[None, :] > first + torch.arange(tokens, device="cuda")[:, None]
    for head in range(heads):
        scores = (q[:, head] @ k[head // group].t()) / math.sqrt(d)
        out[:, head] = torch.softmax(scores.masked_fill(future, float("-inf")), dim=1) @ v[head // group]
    return out.reshape(tokens, heads * d)


def _exact_model(case: dict, seed: int) -> dict:
    inputs = _model_inputs(case, seed)
    hidden, heads, kv_heads, inter = CLASSES[case["class"]]
    palette = _palette()
    weight = {n: _dense(b, s, palette, torch.bfloat16) for n, (b, s) in inputs["weights"].items()}
    decode = case["kind"] == "decode_step"
    first, ids = (case["position"] if decode else 0), inputs["ids"]
    tokens = ids.numel()
    past = (case["layers"], kv_heads, _cached(case), HEAD_DIM)
    keys = inputs["k"].double() if decode else torch.zeros(past, dtype=torch.float64, device="cuda")
    values = inputs["v"].double() if decode else torch.zeros(past, dtype=torch.float64, device="cuda")
    # the rotation's angles as a decoder tabulates them, in float32
    steps = torch.arange(0, HEAD_DIM, 2, device="cuda", dtype=torch.float32) / HEAD_DIM
    angle = torch.arange(first, first + tokens, device="cuda", dtype=torch.float32)[:, None] / (1e6 ** steps)[None, :]
    cos, sin = angle.double().cos()[:, None, :], angle.double().sin()[:, None, :]

    def norm(h, w):
        return h * torch.rsqrt(h.square().mean(-1, keepdim=True) + 1e-6) * w.double()

    def rotate(x):
        lo, hi = x[..., :HEAD_DIM // 2], x[..., HEAD_DIM // 2:]
        return torch.cat([lo * cos - hi * sin, hi * cos + lo * sin], dim=-1)

    h = inputs["embed"][ids].double()
    for layer in range(case["layers"]):
        x = norm(h, inputs["norms"][2 * layer])
        q = rotate((x @ weight["self_attn.q_proj"].t()).view(tokens, heads, HEAD_DIM))
        k = rotate((x @ weight["self_attn.k_proj"].t()).view(tokens, kv_heads, HEAD_DIM))
        v = (x @ weight["self_attn.v_proj"].t()).view(tokens, kv_heads, HEAD_DIM)
        keys[layer, :, first:first + tokens], values[layer, :, first:first + tokens] = k.transpose(0, 1), v.transpose(0, 1)
        seen = first + tokens
        h = h + _attend(q, keys[layer, :, :seen], values[layer, :, :seen], first) @ weight["self_attn.o_proj"].t()
        x = norm(h, inputs["norms"][2 * layer + 1])
        act = torch.nn.functional.silu(x @ weight["mlp.gate_proj"].t()) * (x @ weight["mlp.up_proj"].t())
        h = h + act @ weight["mlp.down_proj"].t()
    x = norm(h, inputs["norms"][-1])
    logits = x[-1:] @ inputs["lm_head"].double().t()
    if decode:
        return {"logits": logits.view(-1), "k": keys, "v": values}
    return {"hidden": x, "logits": logits, "k": keys, "v": values}


@torch.inference_mode()
def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "linear":
        inputs = _linear_inputs(case, seed)
        palette = inputs["palette"] if case["lut"] else _palette()
        y = inputs["x"].double() @ _dense(inputs["blocks"], inputs["scales"], palette, _dtype(case)).t()
        return y + inputs["bias"].double() if case["bias"] else y
    if kind in ("decode_attention", "prompt_attention"):
        inputs = _attention_inputs(case, seed)
        seen, first = (case["position"] + 1, case["position"]) if kind == "decode_attention" else (case["tokens"], 0)
        q = inputs["q"].double().view(-1, case["heads"], HEAD_DIM)
        return _attend(q, inputs["k"][:, :seen].double(), inputs["v"][:, :seen].double(), first)
    if kind == "encode":
        inputs = _encode_inputs(case, seed)
        return {"blocks": None, "scales": inputs["weight"].double().abs().amax(1).clamp_min(1e-12)}
    return _exact_model(case, seed)
