"""The work whose speed is measured: whole calls, single layers and row
operators of the backbone, over the sizes, data types and masks they are used at.

``listed()`` names the cases, ``draw(rng)`` gives one more of the same ranges,
``prepare`` makes what a program holds before the call, ``run`` is one pass
through the public entry points, ``exact`` the same result in 64 bits from plain
torch.  Models are random-initialised from the seed; every tensor has the
distribution its kind has in use (the decay parameters of the linear-attention
layers above all, which decide how far back their state reaches).
"""
import math
import os
import sys

import numpy as np
import torch

PACKAGE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                       "qwendecisioncore.jl_amd")
if PACKAGE not in sys.path:
    sys.path.insert(0, PACKAGE)

from qdc_amd import backbone, config, graphs, ops, weights  # noqa: E402

DEVICE = "cuda:0"
EPS = float(np.float32(1e-6))
# storage of a model: the constructor's dtype and split_gemm_inputs
STORAGE = {"f32": (torch.float32, False), "bf16": (torch.bfloat16, False),
           "mlp": (torch.bfloat16, "mlp"), "all": (torch.bfloat16, "all")}
LAYERS = {"attention": ("full_attention",), "delta": ("linear_attention",),
          "hybrid4": config.hybrid_layer_types(4), "hybrid24": config.hybrid_layer_types(24)}


def listed():
    return [
        # One short prompt scored after another by a small decision model, from
        # recorded graphs: the smallest call, bound by launches and latency.
        _decision("decision_64", 64, "none"),
        # The same with a longer, left-padded prompt of odd length.
        _decision("decision_411_padded", 411, "prefix"),
        # A host batch of padded prompts, one state per prompt (the batched hook).
        _model("prompts_4x300_padded", "last", "0.8b", "hybrid4", "mlp", 4, 300, "prefix"),
        # One full-attention layer over a full batch: prefill of 8 sequences.
        _model("attention_8x2048_bf16", "states", "0.8b", "attention", "bf16", 8, 2048, "none"),
        # The default data type, a ragged length and padding that leaves holes.
        _model("attention_3x777_f32_holes", "states", "0.8b", "attention", "f32", 3, 777, "holes"),
        # One long document of odd length.
        _model("attention_1x6001_bf16", "states", "0.8b", "attention", "bf16", 1, 6001, "none"),
        # One linear-attention layer over a full batch, in the mode that keeps
        # the MLP's inputs at two bf16 terms.
        _model("delta_8x2048_mlp", "states", "0.8b", "delta", "mlp", 8, 2048, "none"),
        # A single padded prompt in the default data type.
        _model("delta_1x777_f32_padded", "states", "0.8b", "delta", "f32", 1, 777, "prefix"),
        # A wider layer with two value heads per key head, odd length, all-bf16.
        _model("delta_2x1501_wide_bf16", "states", "wide", "delta", "bf16", 2, 1501, "none"),
        # Every position of a full batch through the 24-layer model.
        _model("hybrid24_8x2048_mlp", "states", "0.8b", "hybrid24", "mlp", 8, 2048, "none"),
        # Row operators by themselves, as a host program calls them.
        {"name": "residual_norm_4099x1024", "kind": "residual_norm", "rows": 4099, "width": 1024,
         "out": "bf16"},
        {"name": "swiglu_16384x3584_split", "kind": "swiglu", "rows": 16384, "width": 3584,
         "out": "split"},
    ]


def _decision(name, tokens, mask):
    return {"name": name, "kind": "decision", "shape": "decision", "layers": "hybrid4",
            "storage": "f32", "batch": 1, "tokens": tokens, "mask": mask}


def _model(name, kind, shape, layers, storage, batch, tokens, mask):
    return {"name": name, "kind": kind, "shape": shape, "layers": layers, "storage": storage,
            "batch": batch, "tokens": tokens, "mask": mask}


def _log_int(rng, low, high):
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(["decision", "last", "attention", "attention", "delta", "delta", "hybrid",
                       "residual_norm", "swiglu"])
    if kind == "residual_norm":
        return {"kind": kind, "rows": _log_int(rng, 64, 16384),
                "width": rng.choice([256, 1024, 2048]), "out": rng.choice(["f32", "bf16", "split"])}
    if kind == "swiglu":
        return {"kind": kind, "rows": _log_int(rng, 64, 16384),
                "width": rng.choice([512, 3584, 6144]), "out": rng.choice(["f32", "bf16", "split"])}
    mask = rng.choice(["none", "none", "prefix", "holes"])
    if kind == "decision":
        case = _decision("", _log_int(rng, 16, 512), mask)
    elif kind == "last":
        case = _model("", "last", "0.8b", "hybrid4", rng.choice(["f32", "bf16", "mlp", "all"]),
                      rng.randint(1, 8), _log_int(rng, 16, 1024), mask)
    else:
        batch = rng.randint(1, 8)
        tokens = _log_int(rng, 33, min(6001, 16384 // batch))
        layers = "hybrid4" if kind == "hybrid" else kind
        case = _model("", "states", rng.choice(["0.8b", "0.8b", "wide"]), layers,
                      rng.choice(["f32", "bf16", "mlp", "all"]), batch, tokens, mask)
    del case["name"]
    return case


# ------------------------------------------------------------------- inputs --
def _config(case):
    """The shapes of the case's model.  Single layers and short stacks take a
    vocabulary of 4096: the table's size is only seen by the row gather."""
    layers = LAYERS[case["layers"]]
    if case["shape"] == "decision":
        return config.synthetic_inference_config()
    if case["shape"] == "wide":  # 16 / 4 heads of 256, 16 key and 32 value heads of 128
        return config.BackboneConfig(hidden=2048, head_dim=256, heads=16, kv_heads=4,
                                     key_heads=16, value_heads=32, key_dim=128, value_dim=128,
                                     eps=EPS, rope_theta=1e7, rotary_dim=64, layer_types=layers,
                                     intermediate=6144, vocab=4096)
    base = config.qwen35_08b_config().as_dict()
    base.update(layer_types=layers, vocab=248320 if case["layers"] == "hybrid24" else 4096)
    return config.BackboneConfig(**base)


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _weights(case, cfg, seed):
    """Checkpoint tensors on the device in the model's stored dtype."""
    dtype = STORAGE[case["storage"]][0]
    g = _generator(seed)

    def uniform(shape, low, high):
        return torch.empty(shape, device=DEVICE).uniform_(low, high, generator=g)

    out = {}
    for name, shape in weights.all_shapes(cfg).items():
        if name.endswith("A_log"):          # decay rates spread over 1 .. 16
            t = uniform(shape, 1.0, 16.0).log()
        elif name.endswith("dt_bias"):      # time steps spread over 0.001 .. 0.1
            dt = uniform(shape, math.log(1e-3), math.log(1e-1)).exp()
            t = dt + torch.log(-torch.expm1(-dt))
        elif name.endswith("conv1d.weight"):
            t = uniform(shape, -0.5, 0.5)
        else:
            # projections into the residual stream shrink with depth
            deep = name.endswith(("o_proj.weight", "out_proj.weight", "down_proj.weight"))
            std = 0.02 / math.sqrt(2 * len(cfg.layer_types)) if deep else 0.02
            if name.startswith("embed_tokens") and len(cfg.layer_types) > 1:
                std = 0.3   # rows as large as what the layers add to them; a single
                            # layer's result is all but its own output
            t = torch.randn(shape, generator=g, device=DEVICE) * std
            if name.endswith("linear_attn.norm.weight"):
                t += 1.0                    # not zero-centred
        out[name] = t.to(dtype)
    return out


def _sequences(case, cfg, seed):
    """Host ids and 0/1 mask ``[batch, tokens]``."""
    rng = np.random.default_rng(seed)
    shape = (case["batch"], case["tokens"])
    ids = rng.integers(0, cfg.vocab, size=shape)
    mask = np.ones(shape, np.int64)
    if case["mask"] == "prefix":            # left padding of up to a third
        for r in range(shape[0]):
            mask[r, :rng.integers(1, shape[1] // 3 + 2)] = 0
    elif case["mask"] == "holes":
        mask[rng.random(shape) < 0.1] = 0
    mask[:, -1] = 1
    return ids, mask


def _rows(case, seed):
    g = _generator(seed)

    def randn(*shape, scale=1.0):
        return torch.randn(shape, generator=g, device=DEVICE) * scale

    rows, width, out = case["rows"], case["width"], case["out"]
    if case["kind"] == "residual_norm":     # residual stream, layer output, norm weight
        weight = randn(width, scale=0.02)
        return (randn(rows, width), randn(rows, width, scale=0.5),
                weight if out == "f32" else weight.bfloat16())
    packed = randn(rows, 2 * width)         # gate | up of one packed projection
    return (packed.bfloat16() if out == "bf16" else packed,)


def prepare(case, seed):
    if case["kind"] in ("residual_norm", "swiglu"):
        return {"case": case, "rows": _rows(case, seed)}
    cfg = _config(case)
    dtype, split = STORAGE[case["storage"]]
    model = backbone.QwenBackbone.from_weights(_weights(case, cfg, seed), cfg, DEVICE, dtype,
                                               split_gemm_inputs=split)
    ids, mask = _sequences(case, cfg, seed)
    state = {"case": case, "model": model, "ids": ids, "mask": mask}
    if case["kind"] == "decision":
        state["ids"], state["mask"] = ids[0], mask[0]
        state["graphs"] = graphs.LastHiddenGraphs(model)
        state["graphs"].entry(case["tokens"], not bool(mask.all()))   # recorded ahead
    elif case["kind"] == "states":
        state["ids"] = torch.from_numpy(ids.astype(np.int32)).to(DEVICE)
        state["mask"] = (None if case["mask"] == "none"
                         else torch.from_numpy(mask.astype(np.int32)).to(DEVICE))
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "decision":
        return state["graphs"](state["ids"], state["mask"])
    if kind == "last":
        return backbone.batch_backbone_hidden(state["model"], state["ids"], state["mask"])
    if kind == "states":
        return backbone.batch_backbone_states(state["model"], state["ids"], state["mask"])
    out = ops.BF16X2 if case["out"] == "split" else None
    if kind == "residual_norm":
        return ops.native_residual_rms(*state["rows"], EPS, out_dtype=out)
    packed, width = state["rows"][0], case["width"]
    return ops.native_mlp_gate(packed[:, :width], packed[:, width:], out_dtype=out)


# --------------------------------------------------------------- yardsticks --
def work(case):
    """Inputs and weights once, results once; the products a forward cannot do
    without, each input and weight at one term."""
    if case["kind"] in ("residual_norm", "swiglu"):
        n = case["rows"] * case["width"]
        wide = 2 if case["out"] == "bf16" else 4
        if case["kind"] == "swiglu":
            return {"bytes": n * 3 * wide, "flops": 5 * n}
        return {"bytes": n * (12 + wide), "flops": 6 * n}
    cfg = _config(case)
    elem = 4 if case["storage"] == "f32" else 2
    T = case["batch"] * case["tokens"]
    rows = T if case["kind"] == "states" else case["batch"]
    wide = sum(math.prod(s) for n, s in weights.all_shapes(cfg).items()
               if not n.startswith("embed_tokens"))
    nbytes = wide * elem + T * (4 + cfg.hidden * elem) + rows * cfg.hidden * 4
    flops = 0
    for i, kind in enumerate(cfg.layer_types):
        # a call for the last position only needs one row after the last mixing step
        out_rows = rows if i + 1 == len(cfg.layer_types) else T
        flops += 2 * out_rows * 3 * cfg.hidden * cfg.intermediate
        if kind == "full_attention":
            q, kv = cfg.heads * cfg.head_dim, cfg.kv_heads * cfg.head_dim
            pairs = (case["batch"] * case["tokens"] * (case["tokens"] + 1) // 2
                     if out_rows == T else T)
            flops += 2 * cfg.hidden * (out_rows * 3 * q + T * 2 * kv) + 4 * pairs * q
        else:
            kw, vw = cfg.key_heads * cfg.key_dim, cfg.value_heads * cfg.value_dim
            flops += 2 * T * cfg.hidden * (2 * kw + vw) + 4 * out_rows * cfg.hidden * vw
            flops += 6 * T * vw * cfg.key_dim
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """From the error against ``exact`` measured over the listed and some drawn
    cases: fp32 1e-6 .. 3e-6 in models (1.3e-7 in the small decision model), 5e-8
    in row operators; one bf16 layer
    4e-3 .. 7.5e-3, 24 of them 3.6e-3 (their embedding carries more of the
    result); bf16 rows 1.7e-3, of which two implementations share all but ties."""
    if case["kind"] in ("residual_norm", "swiglu"):
        return {"rel": 1e-6 if case["out"] == "f32" else 1e-3}
    if case["kind"] == "decision":
        return {"rel": 1e-6}
    if case["storage"] == "f32":
        return {"rel": 1e-5}
    return {"rel": 1.5e-2 if case["layers"] == "hybrid24" else 1e-2}


# ---------------------------------------------------------- 64-bit reference --
def exact(case, seed):
    if case["kind"] == "residual_norm":
        x, mixed, weight = (t.double() for t in _rows(case, seed))
        total = (x.float() + mixed.float()).double()   # the stored sum is an fp32 value
        normed = _norm(total, weight)
        # a split output holds two terms that only their sum determines
        return x + mixed, None if case["out"] == "split" else normed
    if case["kind"] == "swiglu":
        gate, up = _rows(case, seed)[0].double().split(case["width"], dim=1)
        return None if case["out"] == "split" else torch.nn.functional.silu(gate) * up
    cfg = _config(case)
    W = _weights(case, cfg, seed)
    ids, mask = _sequences(case, cfg, seed)
    states = _forward(cfg, W, torch.from_numpy(ids).to(DEVICE),
                      torch.from_numpy(mask).to(DEVICE).bool())
    if case["kind"] == "states":
        return states
    return states[0, -1] if case["kind"] == "decision" else states[:, -1]


def _norm(x, weight):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * (1.0 + weight)


def _forward(cfg, W, ids, mask):
    h = W["embed_tokens.weight"][ids].double()
    for i, kind in enumerate(cfg.layer_types):
        prefix = f"layers.{i}."
        w = {n[len(prefix):]: t.double() for n, t in W.items() if n.startswith(prefix)}
        x = _norm(h, w["input_layernorm.weight"])
        h = h + (_attention if kind == "full_attention" else _delta)(cfg, w, x, mask)
        x = _norm(h, w["post_attention_layernorm.weight"])
        act = torch.nn.functional.silu(x @ w["mlp.gate_proj.weight"].t())
        h = h + (act * (x @ w["mlp.up_proj.weight"].t())) @ w["mlp.down_proj.weight"].t()
    return _norm(h, W["norm.weight"].double())


def _rotate(cfg, x):
    """Half-split partial rotation of ``[batch, tokens, heads, dim]``; the angles
    are fp32 numbers by the model's definition."""
    half = cfg.rotary_dim // 2
    exponent = np.arange(half, dtype=np.float32) * np.float32(2) / np.float32(cfg.rotary_dim)
    power = (float(np.float32(cfg.rope_theta)) ** exponent.astype(np.float64)).astype(np.float32)
    freq = np.float32(1) / power
    angle = np.arange(x.shape[1], dtype=np.float32)[:, None] * freq
    angle = torch.from_numpy(angle).to(x.device).double()[:, None, :]
    cos, sin = angle.cos(), angle.sin()
    a, b = x[..., :half], x[..., half:2 * half]
    return torch.cat([a * cos - b * sin, b * cos + a * sin, x[..., 2 * half:]], -1)


def _attention(cfg, w, x, mask):
    B, S, _ = x.shape
    H, KV, hd = cfg.heads, cfg.kv_heads, cfg.head_dim
    q, gate = (x @ w["self_attn.q_proj.weight"].t()).view(B, S, H, 2, hd).unbind(3)
    k = (x @ w["self_attn.k_proj.weight"].t()).view(B, S, KV, hd)
    v = (x @ w["self_attn.v_proj.weight"].t()).view(B, S, KV, hd)
    q = _rotate(cfg, _norm(q, w["self_attn.q_norm.weight"]))
    k = _rotate(cfg, _norm(k, w["self_attn.k_norm.weight"]))
    causal = torch.ones(S, S, dtype=torch.bool, device=x.device).tril()
    out = torch.empty(B, S, H, hd, dtype=x.dtype, device=x.device)
    low = -torch.finfo(torch.float32).max
    for b in range(B):
        visible = causal & mask[b]
        for n in range(H):
            g = n // (H // KV)
            scores = q[b, :, n] @ k[b, :, g].t().contiguous() / math.sqrt(hd)
            # a query that sees no kept key spreads evenly over every key
            probs = torch.softmax(scores.masked_fill(~visible, low), -1)
            out[b, :, n] = probs @ v[b, :, g].contiguous()
    out = (out * torch.sigmoid(gate)).reshape(B, S, H * hd)
    return out @ w["self_attn.o_proj.weight"].t()


def _delta(cfg, w, x, mask):
    B, S, _ = x.shape
    KH, kd, VH, vd = cfg.key_heads, cfg.key_dim, cfg.value_heads, cfg.value_dim
    kw = KH * kd
    x = x * mask[..., None]
    mixed = x @ w["linear_attn.in_proj_qkv.weight"].t()
    taps = w["linear_attn.conv1d.weight"][:, 0]
    padded = torch.nn.functional.pad(mixed, (0, 0, taps.shape[1] - 1, 0))
    mixed = sum(padded[:, j:j + S] * taps[:, j] for j in range(taps.shape[1]))
    mixed = torch.nn.functional.silu(mixed)

    def unit(t):
        t = t.reshape(B, S, KH, kd)
        t = t * torch.rsqrt(t.square().sum(-1, keepdim=True) + 1e-6)
        return t.repeat_interleave(VH // KH, dim=2)

    q = unit(mixed[..., :kw]) / math.sqrt(kd)
    k = unit(mixed[..., kw:2 * kw])
    v = mixed[..., 2 * kw:].reshape(B, S, VH, vd)
    beta = torch.sigmoid(x @ w["linear_attn.in_proj_b.weight"].t())
    rate = torch.nn.functional.softplus(x @ w["linear_attn.in_proj_a.weight"].t()
                                        + w["linear_attn.dt_bias"])
    keep = torch.exp(-torch.exp(w["linear_attn.A_log"]) * rate)
    state = torch.zeros(B, VH, vd, kd, dtype=x.dtype, device=x.device)
    out = torch.empty(B, S, VH, vd, dtype=x.dtype, device=x.device)
    for t in range(S):
        state *= keep[:, t, :, None, None]
        u = beta[:, t, :, None] * (v[:, t] - (state * k[:, t, :, None, :]).sum(-1))
        state += u[..., None] * k[:, t, :, None, :]
        out[:, t] = (state * q[:, t, :, None, :]).sum(-1)
    z = (x @ w["linear_attn.in_proj_z.weight"].t()).view(B, S, VH, vd)
    scale = torch.rsqrt(out.square().mean(-1, keepdim=True) + EPS)
    out = out * scale * w["linear_attn.norm.weight"] * torch.nn.functional.silu(z)
    return out.reshape(B, S, VH * vd) @ w["linear_attn.out_proj.weight"].t()
