"""The work a user of this framework has it do, as cases that can be timed and compared.

Five paths, each through its public entry point: an MoE layer with the routing in hand
(``fused_experts``) or from router logits (``fused_moe``), a dense W8A8 linear layer
(``apply_int8_linear``), a dense gated MLP (``w8a8_mlp``) and the re-quantisation of a layer's expert
weights after a policy update (``quantize_expert_weights``).  Layer shapes are those of
``prime_rl_amd.inputs.SHAPES``.  A case is a dict of plain values; tensors are made on the GPU from a
seed.
"""

import math

import torch

import prime_rl_amd as moe

DEV = "cuda:0"
LAYERS = {name: moe.inputs.SHAPES[name] for name in ("qwen3-30b-a3b", "glm-4.5-air", "deepseek-v3")}
# Tokens of one call: from one sequence in decode to a full prefill chunk.
MOST_TOKENS = {"qwen3-30b-a3b": 16384, "glm-4.5-air": 8192, "deepseek-v3": 16384}
RECORD_LAYERS = 4  # layers of the routed-experts record a routed call writes one slice of


def listed():
    return [
        # decode of one sequence: launches, their gaps and the host path
        {"name": "moe_decode_1", "path": "routed", "shape": "qwen3-30b-a3b", "tokens": 1},
        # decode of a small batch: the stream of the routed experts' weights
        {"name": "moe_decode_16", "path": "layer", "shape": "qwen3-30b-a3b", "tokens": 16},
        # a rollout engine's ordinary decode batch, not a multiple of anything
        {"name": "moe_decode_203", "path": "routed", "shape": "qwen3-30b-a3b", "tokens": 203},
        # a prefill chunk
        {"name": "moe_prefill_8192", "path": "layer", "shape": "qwen3-30b-a3b", "tokens": 8192},
        # decode with skewed routing and a shared expert that every token visits
        {"name": "moe_skewed_32", "path": "layer", "shape": "glm-4.5-air", "tokens": 32},
        # a short ragged chunk of the same layer
        {"name": "moe_skewed_517", "path": "layer", "shape": "glm-4.5-air", "tokens": 517},
        # decode of a large model: grouped sigmoid router, routed-experts record
        {"name": "moe_grouped_64", "path": "routed", "shape": "deepseek-v3", "tokens": 64},
        # the largest call: a long prefill of a large model
        {"name": "moe_grouped_16384", "path": "layer", "shape": "deepseek-v3", "tokens": 16384},
        # shared expert / dense layer in decode
        {"name": "mlp_decode_5", "path": "mlp", "tokens": 5, "hidden": 4096, "inter": 1408},
        # the same in prefill
        {"name": "mlp_prefill_4096", "path": "mlp", "tokens": 4096, "hidden": 4096, "inter": 1408},
        # a projection of a mixed prefill and decode batch
        {"name": "linear_333", "path": "linear", "tokens": 333, "n": 4096, "k": 2048},
        # policy update: one layer's bf16 expert weights into the engine's int8 parameters, in place
        {"name": "requantise_layer", "path": "requantise", "experts": 128, "inter": 768, "hidden": 2048},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _multiple(rng, lo, hi, of):
    return max(1, round(_log(rng, lo, hi) / of)) * of


def draw(rng):
    kind = rng.choice(("moe", "moe", "moe", "moe", "dense", "dense", "requantise"))
    if kind == "moe":
        shape = rng.choice(sorted(LAYERS))
        # a shared expert fused as one more expert id comes with the routing, not from the router
        path = "layer" if LAYERS[shape].shared_expert else rng.choice(("layer", "routed"))
        return {"path": path, "shape": shape, "tokens": min(MOST_TOKENS[shape], int(_log(rng, 1, MOST_TOKENS[shape] + 1)))}
    if kind == "dense":
        tokens = int(_log(rng, 1, 8193))
        if rng.random() < 0.5:
            return {"path": "linear", "tokens": tokens, "n": _multiple(rng, 512, 8192, 16), "k": _multiple(rng, 512, 8192, 64)}
        return {"path": "mlp", "tokens": tokens, "hidden": _multiple(rng, 1024, 7168, 64), "inter": _multiple(rng, 512, 8192, 64)}
    return {"path": "requantise", "experts": int(_log(rng, 8, 129)), "inter": _multiple(rng, 512, 1408, 64),
            "hidden": _multiple(rng, 1024, 4096, 64)}


# ---- inputs ---------------------------------------------------------------------------------
def _int8_weights(shape, gen):
    """Normally distributed weights quantised per channel, as a checkpoint's are: the largest of a few
    thousand normal values is about 3.7 standard deviations, which the scale maps to 127."""
    w = torch.empty(shape, dtype=torch.int8, device=DEV)
    flat = w.view(-1)
    part = 1 << 28
    buf = torch.empty(min(part, flat.numel()), dtype=torch.bfloat16, device=DEV)
    for at in range(0, flat.numel(), part):
        n = min(part, flat.numel() - at)
        flat[at:at + n] = buf[:n].normal_(0.0, 127 / 3.7, generator=gen).round_().clamp_(-127, 127)
    return w


def _scales(shape, gen):
    return torch.empty(shape, dtype=torch.float32, device=DEV).uniform_(4e-4, 8e-4, generator=gen)


def _activations(rows, cols, gen):
    return torch.empty((rows, cols), dtype=torch.bfloat16, device=DEV).normal_(generator=gen)


def _logits(shape, tokens, gen, device):
    logits = torch.randn((tokens, shape.E), generator=gen, device=device)
    if shape.routing == "zipf":  # expert popularity falls with rank^-1.2
        ranks = torch.randperm(shape.E, generator=gen, device=device).to(torch.float32) + 1.0
        logits -= 1.2 * ranks.log()
    return logits


def _bias(shape, gen, device):
    return torch.randn((shape.E,), generator=gen, device=device) * 0.1 if shape.routing == "grouped" else None


def _route(shape, tokens, gen, device):
    """``(weights fp32 [tokens, k'], ids int32 [tokens, k'])``, as the layer's router would give them."""
    bias, logits = _bias(shape, gen, device), _logits(shape, tokens, gen, device)
    if shape.routing == "grouped":
        scores = logits.sigmoid()
        choice = scores + bias
        groups = choice.view(tokens, shape.n_group, -1)
        kept = groups.topk(2, dim=-1)[0].sum(-1).topk(shape.topk_group, dim=-1)[1]
        mask = torch.zeros((tokens, shape.n_group), dtype=torch.bool, device=device).scatter_(1, kept, True)
        ids = groups.masked_fill(~mask.unsqueeze(-1), -math.inf).flatten(1).topk(shape.k, dim=-1)[1]
    else:
        scores = logits.softmax(dim=-1)
        ids = scores.topk(shape.k, dim=-1)[1]
    weights = scores.gather(1, ids)
    weights = weights / weights.sum(-1, keepdim=True)
    ids = ids.to(torch.int32)
    if shape.shared_expert:
        ids = torch.cat([ids, torch.full((tokens, 1), shape.E, dtype=torch.int32, device=device)], dim=1)
        weights = torch.cat([weights, torch.ones((tokens, 1), device=device)], dim=1)
    return weights.contiguous(), ids.contiguous()


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    path = case["path"]
    if path in ("layer", "routed"):
        s, tokens = LAYERS[case["shape"]], case["tokens"]
        state = {
            "x": _activations(tokens, s.H, gen),
            "w1": _int8_weights((s.E_total, 2 * s.I, s.H), gen), "w2": _int8_weights((s.E_total, s.H, s.I), gen),
            "w1_scale": _scales((s.E_total, 2 * s.I), gen), "w2_scale": _scales((s.E_total, s.H), gen),
        }
        if path == "layer":
            state["weights"], state["ids"] = _route(s, tokens, gen, DEV)
        else:
            state["bias"], state["logits"] = _bias(s, gen, DEV), _logits(s, tokens, gen, DEV)
            state["record"] = torch.zeros((tokens, RECORD_LAYERS, s.k), dtype=torch.uint8, device=DEV)
        return {"case": case, **state}
    if path == "mlp":
        h, i = case["hidden"], case["inter"]
        return {"case": case, "x": _activations(case["tokens"], h, gen), "w13": _int8_weights((2 * i, h), gen),
                "w13_scale": _scales((2 * i,), gen), "w2": _int8_weights((h, i), gen), "w2_scale": _scales((h,), gen)}
    if path == "linear":
        n, k = case["n"], case["k"]
        return {"case": case, "x": _activations(case["tokens"], k, gen), "w": _int8_weights((n, k), gen), "scale": _scales((n,), gen)}
    e, i, h = case["experts"], case["inter"], case["hidden"]
    bf16 = lambda *shape: torch.empty(shape, dtype=torch.bfloat16, device=DEV).normal_(0.0, 0.02, generator=gen)  # noqa: E731
    out = (torch.empty((e, 2 * i, h), dtype=torch.int8, device=DEV), torch.empty((e, 2 * i), device=DEV),
           torch.empty((e, h, i), dtype=torch.int8, device=DEV), torch.empty((e, h), device=DEV))
    return {"case": case, "gate": bf16(e, i, h), "up": bf16(e, i, h), "down": bf16(e, h, i), "out": out}


# ---- one pass -------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    path = case["path"]
    if path == "layer":
        return moe.fused_experts(state["x"], state["w1"], state["w2"], state["weights"], state["ids"], use_int8_w8a8=True,
                                 per_channel_quant=True, w1_scale=state["w1_scale"], w2_scale=state["w2_scale"])
    if path == "routed":
        s = LAYERS[case["shape"]]
        how = {}
        if s.routing == "grouped":
            how = dict(use_grouped_topk=True, num_expert_group=s.n_group, topk_group=s.topk_group, scoring_func="sigmoid",
                       routed_scaling_factor=2.5, e_score_correction_bias=state["bias"])
        out = moe.fused_moe(state["x"], state["w1"], state["w2"], state["logits"], s.k, True, use_int8_w8a8=True,
                            per_channel_quant=True, w1_scale=state["w1_scale"], w2_scale=state["w2_scale"],
                            routed_experts_out=(state["record"], 1), **how)
        return out, state["record"]
    if path == "mlp":
        return moe.w8a8_mlp(state["x"], state["w13"], state["w13_scale"], state["w2"], state["w2_scale"])
    if path == "linear":
        return moe.apply_int8_linear(state["x"], state["w"], state["scale"])
    return moe.quantize_expert_weights(state["gate"], state["up"], state["down"], out=state["out"])


# ---- what a pass cannot do without, and how close two correct ones come ------------------------
def work(case):
    path = case["path"]
    if path in ("layer", "routed"):
        s, m = LAYERS[case["shape"]], case["tokens"]
        active = _route(s, m, torch.Generator().manual_seed(0), "cpu")[1].unique().numel()  # experts routed to
        routing = m * s.E * 4 + m * s.k if path == "routed" else 8 * m * s.k_total
        return {"bytes": active * (3 * s.I * s.H + 4 * (2 * s.I + s.H)) + 4 * m * s.H + routing, "flops": 6 * m * s.k_total * s.I * s.H}
    if path == "mlp":
        m, h, i = case["tokens"], case["hidden"], case["inter"]
        return {"bytes": 3 * h * i + 4 * (2 * i + h) + 4 * m * h, "flops": 6 * m * h * i}
    if path == "linear":
        m, n, k = case["tokens"], case["n"], case["k"]
        return {"bytes": n * k + 4 * n + 2 * m * (n + k), "flops": 2 * m * n * k}
    e, i, h = case["experts"], case["inter"], case["hidden"]
    return {"bytes": 9 * e * i * h + 4 * e * (2 * i + h), "flops": 0}


def tolerance(case):
    if case["path"] == "requantise":
        return "exact"
    # bf16 results; where activations are quantised a second time, a last-bit difference before that moves a
    # few of them to the next int8 step.  Router scores that agree to fp32 resolution may swap two experts.
    return {"rel": 1e-2, "max": 0.1, "differ": 1e-4}
