"""Workloads of the MoE block, for timing it and comparing its outputs.

A case is one call (or, with `layers` > 1, one pass through several layers' MoE halves) of
`Qwen35MoEModule`, the framework's module: a router, a stack of routed experts in one of the
formats it loads, and usually a shared expert. Shapes:

  c0  hidden 512,  16 experts,  top-2,  intermediate 256, float32 router, no shared expert
  c1  hidden 2048, 256 experts, top-8,  intermediate 512, shared 512
  c2  hidden 4096, 512 experts, top-10, intermediate 1024, shared 1024
  c3  hidden 7168, 256 experts, top-8,  intermediate 2048, shared 2048, sigmoid scores with a
      correction bias, 8 groups of which 4 are kept

Formats: "int4" g64; "int6" g64; "int3-int4" g128 (gate and up int3, down int4); "awq" int4 g64
with per-input-channel activation scales and a clamped activation; "bf16" stacks; "float32"
(activations, scales and router in float32, int4 g32: the dtype of the reference's own checks).
Shared experts are int8 g64, as a bake stores them, or bf16.

Weights are N(0, 0.02) rounded to the nearest code of their group; activations are N(0, 1).
"""

from __future__ import annotations

import math

import torch

from quanta_amd import MoEConfig, Qwen35MoEModule

DEV = "cuda"
BITS = {"int4": (4, 4), "int6": (6, 6), "int3-int4": (3, 4), "awq": (4, 4), "float32": (4, 4),
        "bf16": (16, 16)}
GROUP = {"int4": 64, "int6": 64, "int3-int4": 128, "awq": 64, "float32": 32, "bf16": 0}

C0 = dict(hidden=512, experts=16, top_k=2, inter=256, shared_inter=0, shared="none", gated=False,
          router="softmax", router_dtype="float32")
C1 = dict(hidden=2048, experts=256, top_k=8, inter=512, shared_inter=512, shared="int8", gated=True,
          router="softmax", router_dtype="bf16")
C2 = dict(hidden=4096, experts=512, top_k=10, inter=1024, shared_inter=1024, shared="int8", gated=True,
          router="softmax", router_dtype="bf16")
C3 = dict(hidden=7168, experts=256, top_k=8, inter=2048, shared_inter=2048, shared="bf16", gated=False,
          router="sigmoid-groups", router_dtype="bf16")


def _case(shape, tokens, fmt="int4", *, residual=False, zipf=False, layers=1, **kw):
    return dict(shape, tokens=tokens, format=fmt, residual=residual, zipf=zipf, layers=layers, **kw)


def listed():
    return [
        # the smallest block: launches and host time
        dict(_case(C0, 8), name="c0-8"),
        # the reference's float32 parity configuration, at c0's widths
        dict(_case(C0, 8, "float32"), name="c0-8-float32"),
        # one user's decode step, a small and a large model's layer
        dict(_case(C1, 1), name="c1-1"),
        dict(_case(C2, 1), name="c2-1"),
        # a decode step through several decoder layers' MoE halves (norm and residual included)
        dict(_case(C1, 13, residual=True, layers=4), name="c1-13-step"),
        # batched decode, the block alone; the headline batch
        dict(_case(C2, 32), name="c2-32"),
        # batched decode with DeepSeek's router and an ungated bf16 shared expert
        dict(_case(C3, 16), name="c3-16"),
        # a short prompt: the first sizes above the decode regime, few rows per expert
        dict(_case(C1, 391, residual=True), name="c1-391"),
        # a prompt chunk in int6
        dict(_case(C2, 1000, "int6"), name="c2-1000-int6"),
        # a prompt chunk, gate and up in int3 and down in int4
        dict(_case(C1, 2048, "int3-int4"), name="c1-2048-int3"),
        # a prompt chunk with activation-aware scales
        dict(_case(C2, 512, "awq"), name="c2-512-awq"),
        # a long prompt with skewed expert popularity
        dict(_case(C2, 4096, zipf=True), name="c2-4096-zipf"),
    ]


def _flops(c):
    per = c["top_k"] * 3 * c["inter"] * c["hidden"] + 3 * c["shared_inter"] * c["hidden"] + c["experts"] * c["hidden"]
    return 2.0 * c["layers"] * c["tokens"] * per


def draw(rng):
    """Another case of the same ranges: the shapes above or a generic one, 1 to 4096 tokens."""
    pick = rng.random()
    if pick < 0.1:
        c = dict(C0)
    elif pick < 0.35:
        c = dict(C1)
    elif pick < 0.6:
        c = dict(C2)
    elif pick < 0.7:
        c = dict(C3)
    else:
        c = dict(hidden=128 * rng.randint(6, 40), experts=rng.choice([32, 60, 64, 96, 128, 160]),
                 top_k=rng.randint(2, 8), inter=128 * rng.randint(2, 12), shared_inter=0, shared="none",
                 gated=False, router="softmax", router_dtype="bf16")
        if rng.random() < 0.7:
            c.update(shared_inter=128 * rng.randint(2, 12), shared=rng.choice(["int8", "bf16"]),
                     gated=rng.random() < 0.7)
        if c["experts"] % 8 == 0 and rng.random() < 0.3:
            c["router"] = "sigmoid-groups"
    if c["hidden"] == 512 and c["experts"] == 16:
        return _case(c, int(round(math.exp(rng.uniform(0, math.log(256))))), rng.choice(["int4", "float32"]))
    fmt = rng.choice(["int4", "int4", "int4", "int6", "int3-int4", "awq", "bf16"])
    if fmt == "bf16" and c["hidden"] >= 4096 and c["experts"] >= 256:
        fmt = "int4"
    if fmt == "awq":
        # (the large-batch form of the scaled experts takes intermediate sizes of whole 256-row blocks)
        c["inter"] = max(256, c["inter"] // 256 * 256)
    tokens = int(round(math.exp(rng.uniform(0, math.log(4096)))))
    residual = rng.random() < 0.4
    case = _case(c, tokens, fmt, residual=residual, zipf=not residual and rng.random() < 0.3,
                 layers=rng.choice([1, 1, 1, 2]) if residual and c["hidden"] <= 2048 else 1)
    while _flops(case) > 3.5e11:
        case["tokens"] = case["tokens"] * 2 // 3
    return case


# ----------------------------------------------------------------------------------- inputs


def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed((seed * 1000003 + salt) % (1 << 62))


def _randn(shape, g, std=1.0):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * std


def _pack(codes, bits):
    """Codes [..., n] (int32, n a multiple of 32) -> LSB-first 32-bit words [..., n * bits / 32]."""
    n = codes.shape[-1]
    c = codes.reshape(*codes.shape[:-1], n // 32, 32)
    out = torch.zeros(*c.shape[:-1], bits, dtype=torch.int32, device=c.device)
    for i in range(32):
        w, s = divmod(i * bits, 32)
        out[..., w] |= c[..., i] << s
        if s + bits > 32:
            out[..., w + 1] |= c[..., i] >> (32 - s)
    return out.reshape(*codes.shape[:-1], n * bits // 32)


def _codes(w, bits, group, sdtype):
    """Round-to-nearest affine codes of w [..., n]: (codes int32, scale, bias) per group."""
    g = w.float().reshape(*w.shape[:-1], w.shape[-1] // group, group)
    lo = g.amin(-1)
    s = ((g.amax(-1) - lo) / float((1 << bits) - 1)).to(sdtype)
    b = lo.to(sdtype)
    q = ((g - b.float()[..., None]) / s.float()[..., None]).round_().clamp_(0, (1 << bits) - 1)
    return q.to(torch.int32).reshape(w.shape), s, b


def _stack(E, rows, K, bits, group, g, sdtype=torch.bfloat16):
    """A packed triplet of E experts [rows, K] (bits 16: the bf16 stack itself)."""
    per = max(1, (1 << 27) // (rows * K))
    parts = []
    for e0 in range(0, E, per):
        w = _randn((min(per, E - e0), rows, K), g, 0.02).to(torch.bfloat16)
        if bits < 16:
            q, s, b = _codes(w, bits, group, sdtype)
            parts.append((_pack(q, bits), s, b))
        else:
            parts.append((w,))
        del w
    cat = [torch.cat(p) for p in zip(*parts)]
    if bits == 16:
        return cat[0]
    return {"packed": cat[0], "scale": cat[1], "bias": cat[2], "group_size": group, "bits": bits}


def _layer(c, seed, layer):
    """One layer's parameters, as a loader hands them over."""
    g = _gen(seed, 17 * layer + 1)
    E, H, I, Is = c["experts"], c["hidden"], c["inter"], c["shared_inter"]
    f32 = c["format"] == "float32"
    gb, db = BITS[c["format"]]
    gs = GROUP[c["format"]]
    sdt = torch.float32 if f32 else torch.bfloat16
    p = {}
    gate = _randn((E, H), g, 0.02)
    if c["zipf"]:
        rank = torch.randperm(E, generator=g, device=DEV).float() + 1
        gate[:, 0] = -0.88 * torch.log(rank)
    p["gate"] = gate if f32 or c["router_dtype"] == "float32" else gate.to(torch.bfloat16)
    p["gu"] = _stack(E, 2 * I, H, gb, gs, g, sdt)
    p["dn"] = _stack(E, H, I, db, gs, g, sdt)
    if c["format"] == "awq":
        p["gu"]["awq_scale"] = (2.0 ** _randn((E, 2, H), g, 0.3)).to(torch.bfloat16)
        p["dn"]["awq_scale"] = (2.0 ** _randn((E, I), g, 0.3)).to(torch.bfloat16)
    if c["shared"] != "none":
        for key, shape in (("sg", (Is, H)), ("su", (Is, H)), ("sd", (H, Is))):
            w = _randn(shape, g, 0.02).to(torch.bfloat16)
            if c["shared"] == "int8":
                q, s, b = _codes(w, 8, 64, torch.bfloat16)
                w = {"packed": _pack(q, 8), "scale": s, "bias": b, "group_size": 64, "bits": 8}
            p[key] = w
    p["seg"] = _randn((1, H), g, 0.02).to(torch.bfloat16) if c["gated"] else None
    p["corr"] = _randn((E,), g, 0.01) if c["router"] == "sigmoid-groups" else None
    p["norm"] = (1.0 + _randn((H,), g, 0.1)).to(torch.bfloat16)
    return p


def _x(c, seed):
    x = _randn((c["tokens"], c["hidden"]), _gen(seed, 0))
    if c["zipf"]:
        x[:, 0] = 1.0
    return x if c["format"] == "float32" else x.to(torch.bfloat16)


def _config(c):
    kw = {}
    if c["router"] == "sigmoid-groups":
        kw = dict(scoring_func="sigmoid", n_group=8, topk_group=4, routed_scaling_factor=2.5)
    if c["format"] == "awq":
        kw["swiglu_limit"] = 7.0
    return MoEConfig(c["hidden"], c["experts"], c["top_k"], c["inter"], c["shared_inter"], **kw)


def prepare(case, seed):
    """The layers as a program keeps them (weights set once) and the activations."""
    cfg = _config(case)
    mods, norms = [], []
    for l in range(case["layers"]):
        p = _layer(case, seed, l)
        m = Qwen35MoEModule(cfg, device=DEV)
        m.gate = p["gate"]
        if case["format"] == "bf16":
            m.set_experts(p["gu"], p["dn"])
        else:
            m.set_experts_packed(p["gu"], p["dn"])
        if case["shared"] != "none":
            m.shared_gate_proj, m.shared_up_proj, m.shared_down_proj = p["sg"], p["su"], p["sd"]
        m.shared_expert_gate = p["seg"]
        m.e_score_correction_bias = p["corr"]
        mods.append(m)
        norms.append(p["norm"])
    x = _x(case, seed)
    # decode: one token of each sequence; a prompt: the tokens of one sequence
    x = x[:, None, :] if case["tokens"] <= 128 else x[None]
    return {"mods": mods, "norms": norms, "x": x, "residual": case["residual"]}


def run(state):
    y = state["x"]
    for m, nw in zip(state["mods"], state["norms"]):
        y = m.forward_residual(y, nw) if state["residual"] else m(y)
    return y


# ----------------------------------------------------------------------------------- what it takes


def work(case):
    c = case
    E, H, I, Is, N, k = c["experts"], c["hidden"], c["inter"], c["shared_inter"], c["tokens"], c["top_k"]
    gb, db = BITS[c["format"]]
    # bytes per weight: codes, and a scale and a bias per group
    sb = 0.0 if c["format"] == "bf16" else (8.0 if c["format"] == "float32" else 4.0) / GROUP[c["format"]]
    expert = 2 * I * H * (gb / 8 + sb) + I * H * (db / 8 + sb)
    if c["format"] == "awq":
        expert += 2 * (2 * H + I)
    # distinct experts of N tokens under uniform routing
    distinct = E * (1.0 - (1.0 - k / E) ** N)
    shared = 3 * Is * H * (1 + 4 / 64 if c["shared"] == "int8" else 2)
    wide = 4 if c["format"] == "float32" else 2
    router = E * H * (4 if c["router_dtype"] == "float32" else wide)
    act = 2 * N * H * wide
    return {"bytes": float(c["layers"] * (distinct * expert + shared + router) + act), "flops": _flops(c)}


def tolerance(case):
    # measured against exact(): float32 1.7e-7; one layer in bf16 3.7e-3 to 4.9e-3 (the roundings of
    # gate, up, h and the down rows to bf16); through several layers a rounding that moves a token
    # across a near-tie of the router changes that token's experts (1.5e-2 with 13 tokens)
    if case["format"] == "float32":
        return {"rel": 1e-6}
    return {"rel": 3e-2 if case["layers"] > 1 else 1e-2}


# ----------------------------------------------------------------------------------- in 64 bits


def _weights(v, e=None):
    """The float64 weights of a triplet (or of one expert of a stack), or of a dense matrix."""
    if not isinstance(v, dict):
        return (v if e is None else v[e]).double()
    w, s, b = (v[key] if e is None else v[key][e] for key in ("packed", "scale", "bias"))
    bits, gs = v["bits"], v["group_size"]
    w = w.reshape(*w.shape[:-1], w.shape[-1] // bits, bits).long() & 0xFFFFFFFF
    q = []
    for i in range(32):
        j, sh = divmod(i * bits, 32)
        c = w[..., j] >> sh
        if sh + bits > 32:
            c = c | (w[..., j + 1] << (32 - sh))
        q.append(c & ((1 << bits) - 1))
    q = torch.stack(q, -1).reshape(*w.shape[:-2], -1, gs).double()
    return (s.double()[..., None] * q + b.double()[..., None]).flatten(-2)


def _route(c, p, x):
    logits = x @ p["gate"].double().T
    E, k = c["experts"], c["top_k"]
    if c["router"] == "softmax":
        score = torch.softmax(logits, -1)
        idx = torch.topk(score, k, -1).indices
        scale = 1.0
    else:
        score = torch.sigmoid(logits)
        choice = score + p["corr"].double()
        groups = torch.topk(choice.reshape(-1, 8, E // 8), 2, -1).values.sum(-1)
        keep = torch.zeros_like(groups).scatter_(1, torch.topk(groups, 4, -1).indices, 1.0)
        mask = keep.repeat_interleave(E // 8, -1) > 0
        idx = torch.topk(choice.masked_fill(~mask, -math.inf), k, -1).indices
        scale = 2.5
    w = score.gather(1, idx)
    return idx, w / w.sum(-1, keepdim=True) * scale


def _glu(c, g, u):
    if c["format"] == "awq":
        g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0)
    return torch.nn.functional.silu(g) * u


def exact(case, seed):
    c, I = case, case["inter"]
    x = _x(c, seed).double()
    for l in range(c["layers"]):
        p = _layer(c, seed, l)
        h = x
        if c["residual"]:
            # (a layer's input and its normalised rows are bf16 tensors, which decide the routing)
            x = x.to(torch.bfloat16).double()
            h = p["norm"].double() * x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6)
            h = h.to(torch.bfloat16).double()
        idx, w = _route(c, p, h)
        y = torch.zeros_like(h)
        for e in idx.unique().tolist():
            t, s = (idx == e).nonzero(as_tuple=True)
            gu, a = _weights(p["gu"], e), h[t]
            if c["format"] == "awq":
                sg, su = p["gu"]["awq_scale"][e].double()
                mid = _glu(c, (a / sg) @ gu[:I].T, (a / su) @ gu[I:].T) / p["dn"]["awq_scale"][e].double()
            else:
                mid = _glu(c, a @ gu[:I].T, a @ gu[I:].T)
            y.index_add_(0, t, w[t, s][:, None] * (mid @ _weights(p["dn"], e).T))
        if c["shared"] != "none":
            # (a bake's int8 shared expert is loaded as bf16 weights)
            sg, su, sd = (_weights(p[key]).to(torch.bfloat16).double() for key in ("sg", "su", "sd"))
            out = _glu(c, h @ sg.T, h @ su.T) @ sd.T
            y = y + (torch.sigmoid(h @ p["seg"].double().T) * out if c["gated"] else out)
        x = x + y if c["residual"] else y
    return x[:, None, :] if c["tokens"] <= 128 else x[None]
