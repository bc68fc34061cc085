"""The work that users of this framework have it do, as cases to measure.

Every case runs through the package's public entry points (pocketlm_amd.native)
on tensors that live on the GPU.  The kinds of call, in the order of a token's
way through a model:

  linear      one FP8 block-scaled projection on 1 to 512 activation rows
              (one token, a verifier batch, a prompt chunk), bf16 or fp32 rows
  mlp         the SwiGLU MLP of a shared expert or dense layer, 1 to 512 rows
  moe_step    a DeepSeek-shaped MoE layer from the router's logits, 1 to 8 rows
  moe_routed  the same layer from the router's choices, 1 to 8 rows
  moe_pairs   the routed experts on the (expert, row) pairs of a prompt chunk
  attention   one decode step of the FP8 model's multi-head latent attention
  layer_step  one decode step of a dense decoder layer over its KV cache
  layer_prompt a prompt through a dense decoder layer into a fresh KV cache
  q4_mlp      one token through selected Q4 SwiGLU experts
  lm_head     the top logits of one hidden state over the vocabulary

Sizes are those of the repository's benchmark (DeepSeek-V3 shaped FP8 layers,
a Qwen2.5-7B shaped dense layer) and generic smaller ones.  FP8 weights are
N(0, 0.02) cast to e4m3 with scales uniform in (1e-3, 1e-2), 16-bit weights
N(0, 0.02), activations N(0, 1).
"""

import math

import torch

from pocketlm_amd import formats, native

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed():
    return [
        # the smallest call of a decode step: the latent KV projection of one token
        {"name": "linear_one_token", "kind": "linear", "rows": 576, "cols": 7168, "tokens": 1, "dtype": "bf16"},
        # a speculative verifier's batch through the largest projection
        {"name": "linear_verifier", "kind": "linear", "rows": 7168, "cols": 16384, "tokens": 8, "dtype": "bf16"},
        # a prompt chunk of ragged length through the query up-projection
        {"name": "linear_prompt", "kind": "linear", "rows": 24576, "cols": 1536, "tokens": 509, "dtype": "bf16"},
        # a prompt chunk through the shared expert, with the fp32 rows that callers of the C ABI pass
        {"name": "mlp_prompt", "kind": "mlp", "hidden": 7168, "inter": 2048, "tokens": 256, "dtype": "fp32"},
        # one generated token through a whole MoE layer, router included
        {"name": "moe_one_token", "kind": "moe_step", "hidden": 7168, "inter": 2048, "experts": 256, "top_k": 8,
         "tokens": 1},
        # a verifier's batch through a whole MoE layer
        {"name": "moe_verifier", "kind": "moe_routed", "hidden": 7168, "inter": 2048, "experts": 256, "top_k": 8,
         "tokens": 4},
        # a prompt chunk through the routed experts
        {"name": "moe_prompt", "kind": "moe_pairs", "hidden": 7168, "inter": 2048, "experts": 256, "top_k": 8,
         "tokens": 96, "dtype": "bf16"},
        # one generated token through the FP8 model's attention, some pages into a conversation
        {"name": "attention_one_token", "kind": "attention", "hidden": 7168, "heads": 128, "q_rank": 1536,
         "kv_rank": 512, "nope": 128, "rope": 64, "value": 128, "context": 4096},
        # one generated token through a dense layer
        {"name": "layer_one_token", "kind": "layer_step", "hidden": 3584, "inter": 18944, "heads": 28, "kv_heads": 4,
         "context": 1024, "dtype": "fp16", "biases": True},
        # a short prompt through a dense layer
        {"name": "layer_prompt", "kind": "layer_prompt", "hidden": 3584, "inter": 18944, "heads": 28, "kv_heads": 4,
         "tokens": 120, "dtype": "fp16", "biases": True},
        # one generated token through a Q4 MLP
        {"name": "q4_one_token", "kind": "q4_mlp", "hidden": 3584, "inter": 18944, "selected": 1},
        # the end of a generated token: the vocabulary's largest logits
        {"name": "lm_head", "kind": "lm_head", "vocab": 152064, "hidden": 3584, "top_k": 50, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _step(rng, lo, hi, step):
    """A multiple of step from lo to hi, spread over its logarithm."""
    return max(lo // step, min(hi // step, int(round(_log(rng, lo, hi) / step)))) * step


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "mlp", "moe_step", "moe_routed", "moe_pairs", "attention",
                       "layer_step", "layer_prompt", "q4_mlp", "lm_head"])
    if kind == "linear":
        cols = _step(rng, 512, 16384, 16)
        rows = _log(rng, 128, min(24576, 7168 * 16384 // cols))
        return {"kind": kind, "rows": rows, "cols": cols, "tokens": _log(rng, 1, 512),
                "dtype": rng.choice(["bf16", "bf16", "fp32"])}
    if kind == "mlp":
        return {"kind": kind, "hidden": _step(rng, 1024, 7168, 16), "inter": _step(rng, 512, 2048, 16),
                "tokens": _log(rng, 1, 512), "dtype": rng.choice(["bf16", "bf16", "fp32"])}
    if kind in ("moe_step", "moe_routed"):
        return {"kind": kind, "hidden": _step(rng, 1024, 7168, 128), "inter": _step(rng, 256, 2048, 128),
                "experts": rng.choice([64, 128, 256]), "top_k": rng.choice([4, 6, 8]), "tokens": rng.randint(1, 8)}
    if kind == "moe_pairs":
        return {"kind": kind, "hidden": _step(rng, 1024, 7168, 128), "inter": _step(rng, 256, 2048, 128),
                "experts": rng.choice([32, 64, 96, 160, 256]), "top_k": rng.choice([2, 4, 6, 8]),
                "tokens": _log(rng, 9, 96), "dtype": rng.choice(["bf16", "bf16", "fp32"])}
    if kind == "attention":
        return {"kind": kind, "hidden": _step(rng, 1024, 7168, 128), "heads": rng.choice([16, 32, 64, 128]),
                "q_rank": rng.choice([512, 768, 1536]), "kv_rank": rng.choice([256, 512]), "nope": 128, "rope": 64,
                "value": 128, "context": _log(rng, 16, 4096)}
    if kind in ("layer_step", "layer_prompt"):
        heads, kv_heads, head = rng.choice([(14, 2, 64), (12, 2, 128), (16, 8, 64), (32, 8, 64), (28, 4, 128)])
        case = {"kind": kind, "hidden": heads * head, "inter": _step(rng, 2048, 18944, 64), "heads": heads,
                "kv_heads": kv_heads, "dtype": rng.choice(["fp16", "bf16"]), "biases": rng.random() < 0.5}
        case["context" if kind == "layer_step" else "tokens"] = _log(rng, 16, 8192) if kind == "layer_step" else \
            _log(rng, 9, 120)
        return case
    if kind == "q4_mlp":
        return {"kind": kind, "hidden": _step(rng, 1024, 3584, 16), "inter": _step(rng, 1024, 9472, 16),
                "selected": rng.randint(1, 2)}
    return {"kind": "lm_head", "vocab": rng.randint(32000, 152064), "hidden": _step(rng, 896, 3584, 8),
            "top_k": rng.choice([1, 20, 50, 64]), "dtype": rng.choice(["fp16", "bf16"])}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, scale=1.0, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, scale, generator=g)


def _fp8(g, *shape):
    """e4m3 bytes of N(0, 0.02) and their block scales, uniform in (1e-3, 1e-2)."""
    out = torch.empty(shape, dtype=torch.uint8, device="cuda")
    flat = out.view(-1)
    part = 1 << 28
    for at in range(0, flat.numel(), part):
        n = min(part, flat.numel() - at)
        flat[at:at + n] = _normal(g, (n,), 0.02, torch.float16).to(torch.float8_e4m3fn).view(torch.uint8)
    grid = [*shape[:-2], -(-shape[-2] // 128), -(-shape[-1] // 128)]
    scale = torch.empty(grid, dtype=torch.float32, device="cuda").uniform_(1e-3, 1e-2, generator=g)
    return out, scale


def _wide(weight, scale):
    """The weight that e4m3 bytes and block scales stand for, in 64 bits."""
    rows, cols = weight.shape
    s = scale.double().repeat_interleave(128, 0)[:rows].repeat_interleave(128, 1)[:, :cols]
    return weight.view(torch.float8_e4m3fn).float().double() * s


def _moe_inputs(c, g):
    e, h, i = c["experts"], c["hidden"], c["inter"]
    gate, up, down = _fp8(g, e, i, h), _fp8(g, e, i, h), _fp8(g, e, h, i)
    shared = None
    if c["kind"] != "moe_pairs":
        shared = [*_fp8(g, i, h), *_fp8(g, i, h), *_fp8(g, h, i)]
    x = _normal(g, (c["tokens"], h)).to(DTYPES[c.get("dtype", "bf16")])
    logits = _normal(g, (c["tokens"], e))
    bias = _normal(g, (e,), 0.1)
    return gate, up, down, shared, x, logits, bias


def _expert(weights, e):
    gate, up, down = weights
    return gate[0][e], gate[1][e], up[0][e], up[1][e], down[0][e], down[1][e]


def _route(logits, bias, top_k):
    """DeepSeek-V3's choice of experts: 4 of 8 groups by the sum of their two best biased scores, then the best
    top_k experts; weights normalised, times 2.5, rounded to bf16."""
    score = torch.sigmoid(logits.double())
    choice = score + bias.double()
    groups = choice.view(choice.shape[0], 8, -1)
    best = groups.topk(2, dim=-1).values.sum(-1).topk(4, dim=-1).indices
    keep = torch.zeros(choice.shape[0], 8, dtype=torch.bool, device=choice.device).scatter_(1, best, True)
    masked = groups.masked_fill(~keep[..., None], -math.inf).view_as(choice)
    idx = masked.topk(top_k, dim=-1).indices
    w = score.gather(1, idx)
    return idx, (w / w.sum(-1, keepdim=True) * 2.5).float().to(torch.bfloat16)


def _layer_inputs(c, g):
    dt, h, i = DTYPES[c["dtype"]], c["hidden"], c["inter"]
    kv = h // c["heads"] * c["kv_heads"]
    shapes = [(h, h), (kv, h), (kv, h), (h, h), (i, h), (i, h), (h, i)]
    weights = [_normal(g, s, 0.02).to(dt) for s in shapes]
    norms = [(1 + _normal(g, (h,), 0.1)).to(dt) for _ in range(2)]
    biases = [_normal(g, (n,), 0.1).to(dt) for n in (h, kv, kv)] if c["biases"] else [None] * 3
    x = _normal(g, (c.get("tokens", 1), h)).to(dt)
    cache = [_normal(g, (c.get("context", 0), kv), 0.5).to(dt) for _ in range(2)]
    return x, norms, weights, biases, cache


def _attention_inputs(c, g):
    h, n, r, q = c["hidden"], c["heads"], c["kv_rank"], c["q_rank"]
    shapes = {"q_a": (q, h), "q_b": (n * (c["nope"] + c["rope"]), q), "kv_a": (r + c["rope"], h),
              "o": (h, n * c["value"])}
    fp8 = {name: _fp8(g, *s) for name, s in shapes.items()}
    kv_b = _normal(g, (n * (c["nope"] + c["value"]), r), 0.02)
    norms = [1 + _normal(g, (k,), 0.1) for k in (q, r)]
    angle = c["context"] * 10000.0 ** (-torch.arange(c["rope"] // 2, dtype=torch.float64, device="cuda") * 2 / c["rope"])
    cache = [_normal(g, (c["context"], k)) for k in (r, c["rope"])]
    x = _normal(g, (h,)).to(torch.bfloat16)
    return x, fp8, kv_b, norms, (angle.cos().float(), angle.sin().float()), cache


def prepare(case, seed):
    c, g = case, _gen(seed)
    kind = c["kind"]
    if kind == "linear":
        w, s = _fp8(g, c["rows"], c["cols"])
        return {"case": c, "args": (w, s, _normal(g, (c["tokens"], c["cols"])).to(DTYPES[c["dtype"]]))}
    if kind == "mlp":
        h, i = c["hidden"], c["inter"]
        weights = [*_fp8(g, i, h), *_fp8(g, i, h), *_fp8(g, h, i)]
        return {"case": c, "args": (*weights, _normal(g, (c["tokens"], h)).to(DTYPES[c["dtype"]]))}
    if kind in ("moe_step", "moe_routed", "moe_pairs"):
        gate, up, down, shared, x, logits, bias = _moe_inputs(c, g)
        items = [_expert((gate, up, down), e) for e in range(c["experts"])]
        state = {"case": c, "x": x, "shared": shared, "logits": logits, "bias": bias}
        if kind == "moe_pairs":
            idx, w = _route(logits, bias, c["top_k"])
            rows = torch.arange(c["tokens"], device="cuda").repeat_interleave(c["top_k"])
            return {**state, "items": items, "pairs": (idx.reshape(-1).contiguous(), rows, w.float().reshape(-1))}
        if kind == "moe_routed":
            state["route"] = native.route_deepseek(logits, top_k=c["top_k"], bias=bias, weights_dtype=torch.float32)
        return {**state, "table": native.FP8ExpertTable(items, c["experts"])}
    if kind == "attention":
        x, fp8, kv_b, norms, rope, cache = _attention_inputs(c, g)
        weights = [*fp8["q_a"], *fp8["q_b"], *fp8["kv_a"], kv_b, *fp8["o"], *norms]
        options = dict(previous_kv_cache=cache[0], previous_pe_cache=cache[1], rope_cos=rope[0], rope_sin=rope[1],
                       q_lora_rank=c["q_rank"], kv_lora_rank=c["kv_rank"], num_heads=c["heads"],
                       qk_nope_dim=c["nope"], qk_rope_dim=c["rope"], v_head_dim=c["value"], rms_eps=1e-6,
                       softmax_scale=(c["nope"] + c["rope"]) ** -0.5)
        return {"case": c, "args": (x, *weights), "options": options}
    if kind in ("layer_step", "layer_prompt"):
        x, norms, weights, biases, cache = _layer_inputs(c, g)
        kv = c["hidden"] // c["heads"] * c["kv_heads"]
        options = dict(hidden_size=c["hidden"], intermediate_size=c["inter"], num_heads=c["heads"],
                       num_kv_heads=c["kv_heads"], rms_eps=1e-6, rope_theta=1e6, q_bias=biases[0], k_bias=biases[1],
                       v_bias=biases[2])
        state = {"case": c, "args": (x, *norms, *[native.pack_weight_rows8(w) for w in weights]), "options": options}
        if kind == "layer_step":
            state["session"] = native.NativeKvSession(1, c["context"] + 8, kv, DTYPES[c["dtype"]])
            state["session"].append_committed(0, *cache, c["context"])
        return state
    if kind == "q4_mlp":
        h, i = c["hidden"], c["inter"]
        experts = []
        for _ in range(c["selected"]):
            experts.append([t for s in ((i, h), (i, h), (h, i))
                            for t in formats.quantize_tensor_to_q4(_normal(g, s, 0.02))[:2]])
        route = torch.empty(c["selected"], device="cuda").uniform_(0.1, 1.0, generator=g)
        return {"case": c, "x": _normal(g, (h,)).to(torch.float16), "experts": experts, "route": route}
    dt = DTYPES[c["dtype"]]
    return {"case": c, "x": _normal(g, (c["hidden"],)).to(dt), "w": _normal(g, (c["vocab"], c["hidden"]), 0.02, dt)}


# ---------------------------------------------------------------- one pass

def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "linear":
        return native.fp8_e4m3_block_linear_f32(*state["args"])
    if kind == "mlp":
        return native.fp8_e4m3_block_mlp_f32(*state["args"])
    if kind == "moe_step":
        r = native.fp8_e4m3_block_moe_from_logits(state["table"], state["x"], state["logits"], state["shared"],
                                                  top_k=c["top_k"], bias=state["bias"])
        return {"output": r.output, "routed": r.routed, "shared": r.shared, "indices": r.indices, "weights": r.weights}
    if kind == "moe_routed":
        r = native.fp8_e4m3_block_moe_device_routed_f32(state["table"], state["x"], *state["route"], state["shared"])
        return {"output": r.output, "routed": r.routed, "shared": r.shared}
    if kind == "moe_pairs":
        return native.fp8_e4m3_block_mlp_many_pair_weighted_nosync(state["items"], state["x"], *state["pairs"])
    if kind == "attention":
        out, cache = native.fp8_attention_block_forward(*state["args"], **state["options"])
        return [out, *cache]
    if kind == "layer_step":
        # a drafted token: its cache row is dropped again, so every pass sees the same context
        out = state["session"].dense_layer_decode_packed_rows8(0, *state["args"], **state["options"])
        state["session"].rollback()
        return out
    if kind == "layer_prompt":
        kv = c["hidden"] // c["heads"] * c["kv_heads"]
        session = native.NativeKvSession(1, c["tokens"] + 64, kv, DTYPES[c["dtype"]])
        out = session.dense_layer_prefill_packed_rows8(0, *state["args"], **state["options"])
        keys, values = session.copy_layer(0)
        session.close()
        return [out, keys, values]
    if kind == "q4_mlp":
        return native.q4_moe_selected_forward_u16(state["x"], state["experts"], state["route"],
                                                  hidden_size=c["hidden"], intermediate_size=c["inter"])
    logits, ids = native.lm_head_topk_u16(state["x"], state["w"], top_k=c["top_k"])
    return [logits, ids]


# ---------------------------------------------------------------- what a pass cannot do without

def _fp8_bytes(rows, cols):
    return rows * cols + 4 * -(-rows // 128) * -(-cols // 128)


def _distinct(experts, picks, tokens):
    """Distinct experts that the tokens are expected to pick."""
    return experts * (1 - (1 - picks / experts) ** tokens)


def work(case):
    c = case
    kind = c["kind"]
    xb = 4 if c.get("dtype") == "fp32" else 2
    if kind == "linear":
        n, k, m = c["rows"], c["cols"], c["tokens"]
        return {"bytes": _fp8_bytes(n, k) + xb * m * k + 4 * m * n, "flops": 2 * m * n * k}
    if kind in ("mlp", "moe_step", "moe_routed", "moe_pairs"):
        h, i, m = c["hidden"], c["inter"], c["tokens"]
        expert = 2 * _fp8_bytes(i, h) + _fp8_bytes(h, i)
        if kind == "mlp":
            return {"bytes": expert + xb * m * h + 4 * m * h, "flops": 6 * m * h * i}
        e, k = c["experts"], c["top_k"]
        shared = 0 if kind == "moe_pairs" else 1
        out = 4 if kind == "moe_pairs" else 10
        return {"bytes": (_distinct(e, k, m) + shared) * expert + (xb + out) * m * h + (12 * k + 4 * e * shared) * m,
                "flops": 6 * m * (k + shared) * h * i}
    if kind == "attention":
        h, n, r, q, t = c["hidden"], c["heads"], c["kv_rank"], c["q_rank"], c["context"] + 1
        dims = [(q, h), (n * (c["nope"] + c["rope"]), q), (r + c["rope"], h), (h, n * c["value"])]
        kv_b = n * (c["nope"] + c["value"]) * r
        cache = t * (r + c["rope"])
        return {"bytes": sum(_fp8_bytes(*d) for d in dims) + 4 * kv_b + 8 * cache + 6 * h,
                "flops": 2 * sum(a * b for a, b in dims) + 2 * kv_b + 2 * n * t * (2 * r + c["rope"])}
    if kind in ("layer_step", "layer_prompt"):
        h, i, m, past = c["hidden"], c["inter"], c.get("tokens", 1), c.get("context", 0)
        kv = h // c["heads"] * c["kv_heads"]
        weights = 2 * h * h + 2 * kv * h + 3 * h * i
        seen = m * past + m * (m + 1) / 2
        return {"bytes": 2 * weights + 4 * past * kv + 4 * m * kv + 4 * m * h, "flops": 2 * m * weights + 4 * seen * h}
    if kind == "q4_mlp":
        h, i, s = c["hidden"], c["inter"], c["selected"]
        return {"bytes": s * (3 * h * i / 2 + 4 * i + 2 * h) + 4 * h, "flops": 6 * s * h * i}
    return {"bytes": 2 * c["vocab"] * c["hidden"] + 2 * c["hidden"] + 12 * c["top_k"],
            "flops": 2 * c["vocab"] * c["hidden"]}


def tolerance(case):
    kind = case["kind"]
    if kind == "linear" and case["dtype"] == "bf16":
        return {"rel": 1e-5}  # fp32 sums of exact products
    if kind in ("linear", "mlp", "moe_pairs", "attention"):
        return {"rel": 3e-5}  # fp32 sums, fp32 factors carried as two bf16 (5e-6 to 9e-6 off 64 bits)
    if kind in ("moe_step", "moe_routed"):
        return {"rel": 5e-4, "max": 1e-2}  # the same, and a total whose bf16 may round the other way
    if kind in ("layer_step", "layer_prompt"):
        # four roundings to 16 bits on the way
        return {"rel": 1e-3, "max": 2e-2} if case["dtype"] == "fp16" else {"rel": 8e-3, "max": 0.1}
    if kind == "q4_mlp":
        return {"rel": 1e-3, "max": 1e-2}  # fp16 out
    return {"rel": 1e-5}  # fp32 sums


# ---------------------------------------------------------------- the same in 64 bits

def _mlp64(weights, x):
    gate, up, down = (_wide(weights[2 * k], weights[2 * k + 1]) for k in range(3))
    x = x.double()
    return (torch.nn.functional.silu(x @ gate.T) * (x @ up.T)) @ down.T


def _rms64(x, w, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _pairs_rope64(x, cos, sin):
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)


def _attention64(c, g):
    x, fp8, kv_b, norms, rope, cache = _attention_inputs(c, g)
    n, r = c["heads"], c["kv_rank"]
    w = {name: _wide(*t) for name, t in fp8.items()}
    cos, sin = (t.double() for t in rope)
    q = _rms64(w["q_a"] @ x.double(), norms[0].double())
    q = (w["q_b"] @ q).view(n, c["nope"] + c["rope"])
    kv = w["kv_a"] @ x.double()
    keys = torch.cat([cache[0].double(), _rms64(kv[:r], norms[1].double())[None]])
    pe = torch.cat([cache[1].double(), _pairs_rope64(kv[r:], cos, sin)[None]])
    b = kv_b.double().view(n, c["nope"] + c["value"], r)
    absorbed = torch.einsum("nd,ndr->nr", q[:, :c["nope"]], b[:, :c["nope"]])
    score = absorbed @ keys.T + _pairs_rope64(q[:, c["nope"]:], cos, sin) @ pe.T
    p = torch.softmax(score * (c["nope"] + c["rope"]) ** -0.5, -1)
    heads = torch.einsum("nr,ndr->nd", p @ keys, b[:, c["nope"]:])
    return [w["o"] @ heads.reshape(-1), keys, pe]


def _layer64(c, g):
    x, norms, weights, biases, cache = _layer_inputs(c, g)
    dt, n, nkv = DTYPES[c["dtype"]], c["heads"], c["kv_heads"]
    hd, m, past = c["hidden"] // n, x.shape[0], cache[0].shape[0]
    store = lambda t: t.to(dt).double()  # noqa: E731  (where the layer's storage type holds a value)
    wq, wk, wv, wo, wg, wu, wd = (w.double() for w in weights)
    bq, bk, bv = (0.0 if b is None else b.double() for b in biases)
    x = x.double()
    y = store(_rms64(x, norms[0].double()))
    q, k, v = (y @ wq.T + bq).view(m, n, hd), (y @ wk.T + bk).view(m, nkv, hd), y @ wv.T + bv
    pos = torch.arange(past, past + m, dtype=torch.float64, device="cuda")
    angle = pos[:, None, None] * 1e6 ** (-torch.arange(hd // 2, dtype=torch.float64, device="cuda") * 2 / hd)
    turn = lambda t: torch.cat([t[..., :hd // 2] * angle.cos() - t[..., hd // 2:] * angle.sin(),  # noqa: E731
                                t[..., hd // 2:] * angle.cos() + t[..., :hd // 2] * angle.sin()], -1)
    keys = torch.cat([cache[0].double(), store(turn(k).reshape(m, -1))])
    values = torch.cat([cache[1].double(), store(v)])
    kh = keys.view(-1, nkv, hd).repeat_interleave(n // nkv, 1)
    vh = values.view(-1, nkv, hd).repeat_interleave(n // nkv, 1)
    score = torch.einsum("mnd,tnd->nmt", turn(q), kh) * hd ** -0.5
    late = torch.arange(past + m, device="cuda")[None] > pos[:, None]
    p = torch.softmax(score.masked_fill(late, -math.inf), -1)
    res = x + store(torch.einsum("nmt,tnd->mnd", p, vh).reshape(m, -1) @ wo.T)
    y = store(_rms64(store(res), norms[1].double()))
    out = res + (torch.nn.functional.silu(y @ wg.T) * (y @ wu.T)) @ wd.T
    return out[0] if c["kind"] == "layer_step" else [out, keys, values]


def _q4_64(packed, scales, rows, cols):
    low, high = (packed & 15).to(torch.int8), (packed >> 4).to(torch.int8)
    q = torch.stack([low, high], -1).reshape(rows, cols)
    return torch.where(q > 7, q - 16, q).double() * scales.double()[:, None]


def exact(case, seed):
    c = case
    kind = c["kind"]
    if kind == "attention":
        return _attention64(c, _gen(seed))
    if kind in ("layer_step", "layer_prompt"):
        return _layer64(c, _gen(seed))
    if kind in ("moe_step", "moe_routed", "moe_pairs"):
        gate, up, down, shared, x, logits, bias = _moe_inputs(c, _gen(seed))
        idx, w = _route(logits, bias, c["top_k"])
        out = torch.zeros(x.shape, dtype=torch.float64, device="cuda")
        for e in idx.unique().tolist():
            row, at = torch.where(idx == e)
            out[row] += w[row, at].double()[:, None] * _mlp64(_expert((gate, up, down), e), x[row])
        if kind == "moe_pairs":
            return [out, None]
        extra = _mlp64(shared, x)
        answer = {"output": out + extra, "routed": out, "shared": extra}
        return {**answer, "indices": None, "weights": w.double()} if kind == "moe_step" else answer
    state = prepare(c, seed)
    if kind == "linear":
        w, s, x = state["args"]
        return x.double() @ _wide(w, s).T
    if kind == "mlp":
        return _mlp64(state["args"][:6], state["args"][6])
    if kind == "q4_mlp":
        h, i, x = c["hidden"], c["inter"], state["x"].double()
        out = torch.zeros(h, dtype=torch.float64, device="cuda")
        for route, t in zip(state["route"].double(), state["experts"]):
            act = torch.nn.functional.silu(_q4_64(t[0], t[1], i, h) @ x) * (_q4_64(t[2], t[3], i, h) @ x)
            out += route * (_q4_64(t[4], t[5], h, i) @ act)
        return out
    logits = torch.cat([part.double() @ state["x"].double() for part in state["w"].split(16384)])
    return [logits.topk(c["top_k"]).values, None]
