"""Workloads of the routed expert layer, for timing and for checking.

Each case is a dict of plain values. ``listed()`` holds the standing ones,
``draw(rng)`` makes more of the same ranges, ``prepare`` builds what a program
holds before the call, ``run`` is one pass through the public entry points, and
``exact`` is the same result in 64-bit torch without this package.

Kinds of case (``kind``):
  layer          router logits -> top-k routes -> routed expert layer (inference)
  train          the same under autograd: output and the gradients of tokens,
                 router logits and every LoRA factor
  expert_choice  experts pick tokens; routed layer over [1, E, C] routes
  block          fused router + routed experts + shared expert (one MoE block)
  magi2          multi-head sigmoid routing + swiglu7 experts, bf16 combine
"""

from __future__ import annotations

import math

import torch

from mirai_amd import CompressedGroupedExperts, Magi2GroupedExperts, route_topk
from mirai_amd.block import FusedSparseMoeBlock

# Expert geometries: (hidden, ffn, experts, top_k).
GEOMETRIES = {
    "small": (512, 1024, 8, 2),
    "balanced": (2048, 1408, 64, 4),
    "many": (2048, 768, 128, 8),
    "wide": (3072, 2048, 64, 4),
    "heads": (256, 512, 256, 4),   # per group: 8 heads x 32 experts
}
HEADS = 8

NF4_LEVELS = (
    -1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453,
    -0.28444138169288635, -0.18477343022823334, -0.09105003625154495, 0.0,
    0.07958029955625534, 0.16093020141124725, 0.24611230194568634, 0.33791524171829224,
    0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0,
)


def _case(kind, geometry, tokens, fmt="nf4", rank=16, zipf=0.0):
    return {"kind": kind, "geometry": geometry, "tokens": int(tokens), "fmt": fmt,
            "rank": int(rank), "zipf": float(zipf)}


def listed():
    cases = [
        # A handful of tokens: launches and latency, a part of the experts active.
        ("nf4_T16", _case("layer", "balanced", 16)),
        # A small image: every expert active with a few rows, weights streamed once.
        ("nf4_T256", _case("layer", "balanced", 256)),
        # Unquantised fp32 layer at the size of a test model.
        ("fp32_T512", _case("layer", "small", 512, fmt="fp32", rank=8)),
        # The NF4 + LoRA layer at an ordinary token count, balanced routes.
        ("nf4_T4096", _case("layer", "balanced", 4096)),
        # Skewed routes over many experts: heavy experts beside nearly empty ones.
        ("nf4_zipf_T8192", _case("layer", "many", 8192, rank=8, zipf=1.2)),
        # The headline: a long clip through the NF4 + LoRA layer.
        ("nf4_T32768", _case("layer", "balanced", 32768)),
        # The largest: INT8 experts, a long clip whose token count is not a power of two.
        ("int8_T32760", _case("layer", "wide", 32760, fmt="int8", rank=32)),
        # Adapter training, forward and backward.
        ("train_nf4_T8192", _case("train", "balanced", 8192)),
        # Adapter training on a short odd batch: INT8, a wide adapter, skewed routes.
        ("train_int8_T1023", _case("train", "many", 1023, fmt="int8", rank=64, zipf=1.2)),
        # A whole MoE block without adapters: fused router, NF4 experts, bf16 shared expert.
        ("block_nf4_T4095", _case("block", "balanced", 4095, rank=0)),
        # Expert-choice routes.
        ("choice_nf4_T8192", _case("expert_choice", "balanced", 8192)),
        # Multi-head experts with swiglu7 and the bf16 combine.
        ("magi2_nf4_T1200", _case("magi2", "heads", 1200, rank=0)),
    ]
    return [{"name": name, **case} for name, case in cases]


def draw(rng):
    kind = rng.choices(("layer", "train", "block", "expert_choice", "magi2"),
                       weights=(5, 2, 1, 1, 1))[0]
    if kind == "magi2":
        geometry = "heads"
    elif kind == "layer":
        geometry = rng.choice(("small", "balanced", "many", "wide"))
    else:
        geometry = rng.choice(("balanced", "many"))
    top = {"layer": 32768, "train": 8192, "block": 16384, "expert_choice": 8192,
           "magi2": 8192}[kind]
    low = {"layer": 1, "train": 64, "block": 16, "expert_choice": 64, "magi2": 16}[kind]
    tokens = int(round(math.exp(rng.uniform(math.log(low), math.log(top)))))
    if kind == "layer" and geometry == "small" and rng.random() < 0.5:
        return _case(kind, geometry, min(tokens, 8192), fmt="fp32", rank=8)
    if geometry == "many":  # twice the experts per token
        tokens = max(low, tokens // 2)
    elif geometry == "wide":
        tokens = min(tokens, 24576)
    fmt = rng.choice(("nf4", "nf4", "int8", "bf16"))
    rank = 0 if kind in ("block", "magi2") else rng.choice((8, 16, 32, 64))
    if kind == "layer" and rng.random() < 0.25:
        rank = 0
    zipf = 1.2 if kind in ("layer", "train") and rng.random() < 0.4 else 0.0
    return _case(kind, geometry, tokens, fmt=fmt, rank=rank, zipf=zipf)


# ------------------------------------------------------------------ inputs
def _dims(case):
    return GEOMETRIES[case["geometry"]]


def _capacity(case):
    d, f, E, k = _dims(case)
    return max(1, case["tokens"] * k // E)


def _gen(seed, stream):
    return torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + stream)


def _dense(case, seed, key):
    """Frozen expert weight [E, out, in] ~ N(0, 0.02), bf16 (fp32 for the fp32 layer)."""
    d, f, E, _ = _dims(case)
    shape = (E, d, f) if key == "w2" else (E, f, d)
    g = _gen(seed, {"w1": 1, "w3": 2, "w2": 3}[key])
    dtype = torch.float32 if case["fmt"] == "fp32" else torch.bfloat16
    out = torch.empty(shape, dtype=dtype, device="cuda")
    for a in range(0, E, 16):
        out[a:a + 16] = torch.randn((min(16, E - a), *shape[1:]), generator=g,
                                    device="cuda") * 0.02
    return out


def _factors(case, seed):
    """LoRA factors {key: (A [E, r, in], B [E, out, r])} ~ N(0, 0.02), fp32."""
    d, f, E, _ = _dims(case)
    r, out = case["rank"], {}
    if r == 0:
        return out
    g = _gen(seed, 4)
    for key, (o, i) in (("w1", (f, d)), ("w3", (f, d)), ("w2", (d, f))):
        out[key] = (torch.randn((E, r, i), generator=g, device="cuda") * 0.02,
                    torch.randn((E, o, r), generator=g, device="cuda") * 0.02)
    return out


def _alpha(case):
    return 32.0 if case["rank"] == 32 else 16.0


def _tokens(case, seed, shape):
    dtype = torch.float32 if case["fmt"] == "fp32" else torch.bfloat16
    return torch.randn(shape, generator=_gen(seed, 5), device="cuda").to(dtype)


def _logits(case, seed):
    """Router logits [T, E] ~ N(0, 1), with a Zipf-ranked bias for skewed routes."""
    E, g = _dims(case)[2], _gen(seed, 6)
    logits = torch.randn((case["tokens"], E), generator=g, device="cuda")
    if case["zipf"]:
        rank = torch.randperm(E, generator=g, device="cuda").float()
        logits = logits - 1.5 * case["zipf"] * torch.log(rank + 1.0)
    return logits


def _choice_routes(case, seed):
    """Every expert takes its capacity of tokens with the highest scores."""
    probs = torch.softmax(_logits(case, seed), dim=1)
    top = torch.topk(probs.t(), _capacity(case), dim=1)
    return top.values.unsqueeze(0).contiguous(), top.indices.unsqueeze(0).contiguous()


def _router(case, seed):
    """Router weight [E, d] and selection bias [E]."""
    d, _, E, _ = _dims(case)
    g = _gen(seed, 7)
    return (torch.randn((E, d), generator=g, device="cuda") * 0.02,
            torch.randn(E, generator=g, device="cuda") * 0.01)


def _shared(case, seed):
    """Shared expert weights gate, up [f, d], down [d, f], bf16."""
    d, f, _, _ = _dims(case)
    g = _gen(seed, 8)
    return [(torch.randn(s, generator=g, device="cuda") * 0.02).to(torch.bfloat16)
            for s in ((f, d), (f, d), (d, f))]


def _head_logits(case, seed):
    """Per-head router logits [H, S, E / H] and selection bias [H, E / H]."""
    n = _dims(case)[2] // HEADS
    g = _gen(seed, 9)
    return (torch.randn((HEADS, case["tokens"], n), generator=g, device="cuda"),
            torch.randn((HEADS, n), generator=g, device="cuda") * 0.05)


def _upstream(case, seed):
    d = _dims(case)[0]
    return torch.randn((case["tokens"], d), generator=_gen(seed, 10),
                       device="cuda").to(torch.bfloat16)


# ----------------------------------------------------------------- the path
def _experts(case, seed):
    m = CompressedGroupedExperts.from_empty(
        num_experts=_dims(case)[2], quant_format=case["fmt"],
        expert_weight_access="fused_kernel", expert_dequant_chunk_size=16)
    for key in ("w1", "w3", "w2"):
        m.load_dense_weight(key, _dense(case, seed, key))
    for key, (a, b) in _factors(case, seed).items():
        ad = m.attach_expert_lora(tensor_name=key, adapter_name="adapter", rank=case["rank"],
                                  alpha=_alpha(case))
        with torch.no_grad():
            ad.lora_a.copy_(a)
            ad.lora_b.copy_(b)
    return m


def prepare(case, seed):
    d, f, E, k = _dims(case)
    T, kind = case["tokens"], case["kind"]
    if kind == "magi2":
        groups = {key: _dense(case, seed, key).transpose(1, 2).contiguous()
                  for key in ("w1", "w3", "w2")}
        logits, bias = _head_logits(case, seed)
        return {"kind": kind, "top_k": k, "x": _tokens(case, seed, (T, HEADS, d)),
                "logits": logits, "bias": bias,
                "experts": Magi2GroupedExperts.from_dense(
                    groups["w1"], groups["w3"], groups["w2"], num_heads=HEADS,
                    quant_format=case["fmt"])}
    state = {"kind": kind, "top_k": k, "x": _tokens(case, seed, (T, d))}
    if kind == "block":
        blk = FusedSparseMoeBlock(d, 4 * d, E, k, f, "sigmoid", True, None, None, 1.0, 1,
                                  quant_format=case["fmt"]).to("cuda")
        blk.experts = _experts(case, seed)
        blk.shared_experts.to(torch.bfloat16)
        weight, bias = _router(case, seed)
        mlp = blk.shared_experts
        with torch.no_grad():
            blk.router.weight.copy_(weight)
            blk.router.e_score_correction_bias.copy_(bias)
            for lin, w in zip((mlp.gate_proj, mlp.up_proj, mlp.down_proj), _shared(case, seed)):
                lin.weight.copy_(w)
        blk.requires_grad_(False)
        return {**state, "x": state["x"].unsqueeze(0), "block": blk}
    state["experts"] = _experts(case, seed)
    if kind == "expert_choice":
        state["scores"], state["indices"] = _choice_routes(case, seed)
        return state
    state["logits"] = _logits(case, seed)
    if kind == "train":
        state["upstream"] = _upstream(case, seed)
        state["x"].requires_grad_(True)
        state["logits"].requires_grad_(True)
    return state


def run(state):
    kind, x, k = state["kind"], state["x"], state["top_k"]
    if kind == "train":
        m = state["experts"]
        idx, scores = route_topk(state["logits"], k)
        out = m.run_direct_routed(x, scores, idx)
        factors = [p for key in ("w1", "w3", "w2")
                   for p in (m.expert_lora[key].lora_a, m.expert_lora[key].lora_b)]
        grads = torch.autograd.grad(out, [x, state["logits"], *factors], state["upstream"])
        return [out.detach(), *grads]
    with torch.no_grad():
        if kind == "layer":
            idx, scores = route_topk(state["logits"], k)
            return state["experts"].run_direct_routed(x, scores, idx)
        if kind == "expert_choice":
            return state["experts"].run_expert_choice_routed(
                x, state["scores"], state["indices"], tokens_per_sample=int(x.shape[0]))
        if kind == "block":
            return state["block"](x)
        return state["experts"](x, state["logits"], top_k=k, score_func="sigmoid",
                                expert_bias=state["bias"], route_scale=1.0)


# --------------------------------------------------------------- accounting
def _active(case, rows):
    """Expected number of experts that any of the routed rows reaches."""
    E = _dims(case)[2]
    if case["zipf"]:
        p = [(e + 1.0) ** (-1.5 * case["zipf"]) for e in range(E)]
    else:
        p = [1.0] * E
    total = sum(p)
    return sum(1.0 - math.exp(-rows * q / total) for q in p)


def work(case):
    d, f, E, k = _dims(case)
    T, r, kind = case["tokens"], case["rank"], case["kind"]
    tok = T * HEADS if kind == "magi2" else T
    rows = _capacity(case) * E if kind == "expert_choice" else tok * k
    act = 4 if case["fmt"] == "fp32" else 2
    per_weight = {"nf4": 0.5 + 2.0 / 64, "int8": 1.0, "bf16": 2.0, "fp32": 4.0}[case["fmt"]]
    expert = 3 * d * f * per_weight + 3 * r * (d + f) * 4
    nbytes = _active(case, rows) * expert + 2 * tok * d * act
    flops = 2 * rows * 3 * d * f + 2 * rows * r * 3 * (d + f)
    if kind == "expert_choice":
        nbytes += rows * 12
    elif kind == "magi2":
        nbytes += tok * (E // HEADS) * 4
    elif kind == "block":
        nbytes += E * d * 4 + 3 * d * f * 2
        flops += 2 * T * d * E + 2 * T * 3 * d * f
    else:
        nbytes += T * E * 4
    if kind == "train":
        # Backward: dX through the frozen weights (as many products as the
        # forward), and per factor both its gradient and the step through it;
        # upstream in, token and logit gradients and the factors' gradients out.
        flops += 2 * rows * 3 * d * f + 4 * rows * r * 3 * (d + f)
        nbytes += 2 * T * d * 2 + T * E * 4 + E * 3 * r * (d + f) * 4
    return {"bytes": int(nbytes), "flops": int(flops)}


def tolerance(case):
    # bf16 layers: the roundings of gate, up, h, y, the output and the factors
    # leave a result 4.4e-3 to 5.4e-3 from the 64-bit one (measured, every kind
    # of case). fp32: split bf16 planes hold a weight to 2^-16, 8.1e-6 measured.
    # About four times that is stated.
    if case["fmt"] == "fp32":
        return {"rel": 3.5e-5, "max": 1e-3}
    return {"rel": 2e-2, "max": 0.3}


# ------------------------------------------------------------ 64-bit result
def _stored(case, w):
    """The values a stored weight [out, in] stands for, in 64 bits: NF4 blocks of
    64 along a row (bf16 absmax, bf16(level * absmax)), INT8 per row (bf16 scale,
    bf16(q * scale)), else the tensor itself."""
    v = w.float()
    if case["fmt"] == "nf4":
        levels = torch.tensor(NF4_LEVELS, dtype=torch.float32, device=v.device)
        blocks = v.reshape(-1, 64)
        absmax = blocks.abs().amax(dim=1, keepdim=True)
        scaled = torch.where(absmax > 0, blocks / absmax, torch.zeros_like(blocks))
        codes = (scaled.unsqueeze(2) - levels).abs().argmin(dim=2)
        v = (levels[codes] * absmax).to(torch.bfloat16).reshape(v.shape)
    elif case["fmt"] == "int8":
        scale = (v.abs().amax(dim=1, keepdim=True) / 127.0).clamp_min(1e-30)
        scale = scale.to(torch.bfloat16).float()
        q = torch.clamp(torch.round(v / scale), -127.0, 127.0)
        v = (q * scale).to(torch.bfloat16)
    return v.double()


def _mlp(x, w, lora, scale, act):
    """One expert in 64 bits: w and lora by role (gate, up, down)."""
    def proj(v, i):
        out = v @ w[i].t()
        if lora[i] is not None:
            out = out + scale * ((v @ lora[i][0].t()) @ lora[i][1].t())
        return out

    g, u = proj(x, 0), proj(x, 1)
    if act == "swiglu7":
        g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0)
        h = g * torch.sigmoid(1.702 * g) * (u + 1.0)
    else:
        h = torch.nn.functional.silu(g) * u
    return proj(h, 2)


def _routed(case, seed, x, idx, scores, act="silu", upstream=None):
    """sum over a row's routes of score * expert(x), [N, d] in 64 bits; with an
    upstream gradient also (grad x, grad scores, factor gradients by key)."""
    E, r = _dims(case)[2], case["rank"]
    keys = ("w1", "w3", "w2")
    dense = [_dense(case, seed, key) for key in keys]
    factors = _factors(case, seed)
    scale = _alpha(case) / r if r else 0.0
    out = torch.zeros(x.shape, dtype=torch.float64, device=x.device)
    gx, gs = torch.zeros_like(out), torch.zeros_like(scores)
    gf = {key: [torch.zeros(t.shape, dtype=torch.float64, device=x.device)
                for t in factors[key]] for key in factors}
    for e in range(E):
        row, slot = torch.nonzero(idx == e, as_tuple=True)
        if row.numel() == 0:
            continue
        w = [_stored(case, t[e]) for t in dense]
        lora = [[t[e].double() for t in factors[key]] if r else None for key in keys]
        xe, se = x[row], scores[row, slot].unsqueeze(1)
        if upstream is None:
            out.index_add_(0, row, _mlp(xe, w, lora, scale, act) * se)
            continue
        leaves = [xe, se, *[t for pair in lora for t in pair]]
        for t in leaves:
            t.requires_grad_(True)
        y = _mlp(xe, w, lora, scale, act) * se
        grads = torch.autograd.grad(y, leaves, upstream[row])
        out.index_add_(0, row, y.detach())
        gx.index_add_(0, row, grads[0])
        gs[row, slot] = grads[1].squeeze(1)
        for i, key in enumerate(keys):
            gf[key][0][e], gf[key][1][e] = grads[2 + 2 * i], grads[3 + 2 * i]
    return out, gx, gs, gf


def exact(case, seed):
    d, f, E, k = _dims(case)
    T, kind = case["tokens"], case["kind"]
    if kind == "magi2":
        x = _tokens(case, seed, (T * HEADS, d)).double()
        logits, bias = _head_logits(case, seed)
        s = torch.sigmoid(logits.double())
        pick = torch.topk(s + bias.double().unsqueeze(1), k, dim=2).indices
        p = torch.gather(s, 2, pick)
        p = p / p.sum(dim=2, keepdim=True).clamp_min(1e-12)
        heads = torch.arange(HEADS, device=pick.device).view(HEADS, 1, 1) * (E // HEADS)
        idx = (pick + heads).permute(1, 0, 2).reshape(T * HEADS, k)
        out = _routed(case, seed, x, idx, p.permute(1, 0, 2).reshape(T * HEADS, k), "swiglu7")[0]
        return out.view(T, HEADS, d)
    x = _tokens(case, seed, (T, d)).double()
    if kind == "expert_choice":
        scores, picked = _choice_routes(case, seed)
        # One row per (expert, slot), then summed into its token.
        C = _capacity(case)
        rows = picked.reshape(-1)
        idx = torch.arange(E, device=rows.device).repeat_interleave(C).unsqueeze(1)
        y = _routed(case, seed, x[rows], idx, scores.reshape(-1, 1).double())[0]
        return torch.zeros_like(x).index_add_(0, rows, y)
    if kind == "block":
        weight, bias = _router(case, seed)
        s = torch.sigmoid(x @ weight.double().t())
        idx = torch.topk(s + bias.double(), k, dim=1).indices
        top = torch.gather(s, 1, idx)
        out = _routed(case, seed, x, idx, top / top.sum(dim=1, keepdim=True))[0]
        shared = [w.double() for w in _shared(case, seed)]
        return (out + _mlp(x, shared, [None] * 3, 0.0, "silu")).unsqueeze(0)
    logits = _logits(case, seed).double()
    top, idx = torch.topk(logits, k, dim=1)
    scores = torch.softmax(top, dim=1)  # softmax over all, renormalised over the picks
    if kind == "layer":
        return _routed(case, seed, x, idx, scores)[0]
    out, gx, gs, gf = _routed(case, seed, x, idx, scores, upstream=_upstream(case, seed).double())
    # The picked scores' softmax Jacobian; logits that were not picked cancel out.
    gl = scores * (gs - (gs * scores).sum(dim=1, keepdim=True))
    glogits = torch.zeros_like(logits).scatter_(1, idx, gl)
    return [out, gx, glogits, *[t for key in ("w1", "w3", "w2") for t in gf[key]]]
