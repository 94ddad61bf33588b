"""Timed cases of the routed-expert path: what a serving program asks of this package.

Shapes are the ones the configurations, tests and bench.py use: 256 routed
experts of hidden size 4096 and intermediate size 2048 in MXFP4, top-6 or top-8,
and the smaller expert shapes of the tests. Expert popularity is Zipf(1.1), as
in bench.py; weights are resident in HBM in the MFMA-tiled layout the slot cache
stores, except in the offload case, which copies them from pinned host memory.
"""

import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "deepseek-v4-flash-offload_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import npu_ops  # noqa: E402
import offload  # noqa: E402
from dsv4_hip import ops, PROFILE_A4W4, PROFILE_BF16, PROFILE_BF16_PURE  # noqa: E402

PROFILES = {"bf16": PROFILE_BF16, "a4w4": PROFILE_A4W4, "pure": PROFILE_BF16_PURE}
ZIPF_S = 1.1
SWIGLU_LIMIT = 10.0
ROUTED_SCALE = 1.5


def _layer(name, tokens, topk, profile, **over):
    case = {"name": name, "kind": "layer", "tokens": tokens, "topk": topk, "profile": profile, "experts": 256,
            "hidden": 4096, "inter": 2048, "route": False, "shared": False, "tiled": True}
    case.update(over)
    return case


def listed():
    return [
        # one sequence being generated: router, routed experts and the FP8 shared expert in one call
        _layer("routed_1_shared", 1, 6, "bf16", route=True, shared=True),
        # a small decode batch (the workload of bench.py)
        _layer("decode_8", 8, 8, "bf16"),
        # a decode batch of a serving engine in the 4-bit activation profile
        _layer("decode_64_a4w4", 64, 8, "a4w4"),
        # a large decode batch, ragged against every tile
        _layer("batch_203", 203, 8, "bf16"),
        # a short prompt in the variant without activation quantisation
        _layer("prefill_509_pure", 509, 6, "pure"),
        # an ordinary prompt chunk
        _layer("prefill_2048", 2048, 8, "bf16"),
        # a long prompt of odd length in the 4-bit activation profile
        _layer("prefill_6007_a4w4", 6007, 6, "a4w4"),
        # the largest chunk bench.py runs
        _layer("prefill_16384", 16384, 8, "bf16"),
        # the router of a prompt chunk by itself, as the offload path calls it before it acquires experts
        {"name": "route_2048", "kind": "route", "tokens": 2048, "topk": 8, "experts": 256, "hidden": 4096},
        # an expert's w1, w2 and w3 to bf16, as a miss of the bf16 expert cache does
        {"name": "dequant_expert", "kind": "dequant", "hidden": 4096, "inter": 2048, "tiled": True},
        # activations of a prompt chunk quantised by the stand-alone operators (FP8 per 128, MXFP4 per 32)
        {"name": "act_quant_4096", "kind": "quant", "tokens": 4096, "hidden": 4096, "rule": "ocp_floor"},
        # two layers of a decode step whose experts all miss the slot cache (bound by the host link)
        {"name": "offload_step", "kind": "offload", "tokens": 8, "topk": 8, "experts": 256, "hidden": 4096,
         "inter": 2048, "pool": 16, "layers": 2},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(["layer", "route", "dequant", "quant", "offload"], [12, 2, 1, 1, 1])[0]
    if kind == "layer":
        profile = rng.choice(["bf16", "bf16", "a4w4", "pure"])
        route = rng.random() < 0.3
        experts, hidden, inter = rng.choice([(256, 4096, 2048)] * 4 + [(128, 2048, 1024), (64, 4096, 1024)])
        return {"kind": kind, "tokens": _log_int(rng, 1, 64 if route else 8192 if profile == "pure" else 16384),
                "topk": rng.choice([6, 8]), "profile": profile, "experts": experts, "hidden": hidden, "inter": inter,
                "route": route, "shared": route and profile == "bf16" and rng.random() < 0.5,
                "tiled": rng.random() < 0.85}
    if kind == "route":
        return {"kind": kind, "tokens": _log_int(rng, 1, 16384), "topk": rng.choice([6, 8]),
                "experts": rng.choice([64, 128, 256]), "hidden": rng.choice([2048, 4096])}
    if kind == "dequant":
        return {"kind": kind, "hidden": rng.choice([1024, 2048, 4096]), "inter": 256 * rng.randint(2, 12),
                "tiled": rng.random() < 0.5}
    if kind == "quant":
        return {"kind": kind, "tokens": _log_int(rng, 8, 16384), "hidden": rng.choice([2048, 4096]),
                "rule": rng.choice(["ocp_floor", "ceil_div6"])}
    return {"kind": kind, "tokens": rng.randint(2, 16), "topk": 8, "experts": 256, "hidden": 4096,
            "inter": rng.choice([1024, 2048]), "pool": rng.randint(8, 16), "layers": 2}


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------
def _gen(seed, stream):
    return torch.Generator(device="cuda").manual_seed(1_000_003 * int(seed) + stream)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _packed(g, *shape):
    """[..., N, K] MXFP4: uniform E2M1 nibbles, E8M0 bytes 117..127."""
    *lead, n, k = shape
    codes = torch.randint(0, 256, (*lead, n, k // 2), dtype=torch.uint8, generator=g, device="cuda")
    scales = torch.randint(117, 128, (*lead, n, k // 32), dtype=torch.uint8, generator=g, device="cuda")
    return codes, scales


def _experts(seed, n, hidden, inter):
    """n experts' packed tensors in the checkpoint layout, stacked over the experts."""
    g = _gen(seed, 1)
    w = {}
    for name, rows, cols in (("w1", inter, hidden), ("w3", inter, hidden), ("w2", hidden, inter)):
        w[name + "p"], w[name + "s"] = _packed(g, n, rows, cols)
    return w


def _table(w, experts, tiled):
    """Device pointer table over the experts stacked in w."""
    if tiled:
        w = {k: ops.tile_weights(v.view(-1, v.shape[-1])).view(v.shape) if k.endswith("p") else v for k, v in w.items()}
    return ops.expert_table({e: {k: v[e] for k, v in w.items()} for e in range(experts)}, experts, "cuda:0", tiled=tiled)


def _routing(seed, tokens, topk, experts):
    """(ids int32 [T, K], weights fp32 [T, K]): K distinct experts per token, Zipf popularity."""
    g = _gen(seed, 2)
    p = torch.arange(1, experts + 1, device="cuda", dtype=torch.float32) ** -ZIPF_S
    noise = -torch.log(-torch.log(torch.rand(tokens, experts, generator=g, device="cuda").clamp(1e-12, 1 - 1e-7)))
    ranks = torch.topk(torch.log(p / p.sum()) + noise, topk, dim=1).indices
    perm = torch.randperm(experts, generator=g, device="cuda")
    w = torch.softmax(_normal(g, tokens, topk), 1)
    return perm[ranks].to(torch.int32).contiguous(), w


def _gate(seed, experts, hidden):
    """(gate weight fp32 [E, D], score correction bias fp32 [E])."""
    g = _gen(seed, 3)
    w = _normal(g, experts, hidden) * hidden ** -0.5
    bias = -0.1 * torch.log(torch.randperm(experts, generator=g, device="cuda").float() + 1.0)
    return w, bias


def _activations(seed, tokens, hidden):
    return _normal(_gen(seed, 4), tokens, hidden).to(torch.bfloat16)


def _shared(seed, hidden, inter):
    """The shared expert as checkpoints hold it: E4M3 codes with 128x128 E8M0 block scales."""
    g = _gen(seed, 5)
    out = {}
    for name, n, k in (("w1", inter, hidden), ("w3", inter, hidden), ("w2", hidden, inter)):
        w = _normal(g, n, k) * 2.0 ** -6
        amax = w.abs().view(n // 128, 128, k // 128, 128).amax(dim=(1, 3))
        e = torch.ceil(torch.log2(amax / 448.0))
        s = torch.exp2(e).repeat_interleave(128, 0).repeat_interleave(128, 1)
        out[name] = (w / s).to(torch.float8_e4m3fn)
        out[name + "s"] = (e + 127).to(torch.uint8)
    return out


def _offload_ids(case, layer):
    """[T, K] ids over the layer's registered experts (the even expert ids), every one of them picked."""
    t, k, pool = case["tokens"], case["topk"], case["pool"]
    flat = (np.arange(t * k) + layer) % pool
    return torch.from_numpy((2 * flat).astype(np.int32).reshape(t, k))


# ---------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "layer":
        E, D, I = case["experts"], case["hidden"], case["inter"]
        s["x"] = _activations(seed, case["tokens"], D)
        s["table"] = _table(_experts(seed, E, D, I), E, case["tiled"])
        s["runner"] = ops.LayerRunner("cuda:0", E, D, I)
        if case["route"]:
            s["gate"], s["bias"] = _gate(seed, E, D)
            s["shared"] = None
            if case["shared"]:
                sh = _shared(seed, D, I)
                s["shared"] = ops.prepare_shared_expert(*[sh[k] for k in ("w1", "w1s", "w3", "w3s", "w2", "w2s")])
        else:
            s["ids"], s["w"] = _routing(seed, case["tokens"], case["topk"], E)
    elif kind == "route":
        s["x"] = _activations(seed, case["tokens"], case["hidden"])
        s["gate"], s["bias"] = _gate(seed, case["experts"], case["hidden"])
    elif kind == "dequant":
        w = _experts(seed, 1, case["hidden"], case["inter"])
        s["pairs"] = [(ops.tile_weights(w[n + "p"][0]) if case["tiled"] else w[n + "p"][0], w[n + "s"][0])
                      for n in ("w1", "w2", "w3")]
    elif kind == "quant":
        s["x"] = _activations(seed, case["tokens"], case["hidden"])
    else:
        s["bank"] = offload.ExpertBank(1, "cuda:0")
        s["bank"].packed_capacity = case["pool"]  # one layer's experts: the next layer's evict them
        for lay in range(case["layers"]):
            w = {k: v.cpu() for k, v in _experts(seed + 7919 * lay, case["pool"], case["hidden"], case["inter"]).items()}
            for i in range(case["pool"]):
                s["bank"].register(lay, 2 * i, *[w[k][i] for k in ("w1p", "w1s", "w2p", "w2s", "w3p", "w3s")])
        s["x"] = _activations(seed, case["tokens"], case["hidden"])
        s["ids"] = [_offload_ids(case, lay).cuda() for lay in range(case["layers"])]
        s["w"] = torch.softmax(_normal(_gen(seed, 2), case["tokens"], case["topk"]), 1)
        s["runner"] = ops.LayerRunner("cuda:0", case["experts"], case["hidden"], case["inter"])
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "layer":
        if case["route"]:
            y, w, ids = s["runner"].forward_routed(s["x"], s["gate"], case["topk"], s["table"], bias=s["bias"],
                                                   scale=ROUTED_SCALE, profile=PROFILES[case["profile"]],
                                                   swiglu_limit=SWIGLU_LIMIT, shared=s["shared"])
            return {"y": y, "weights": w, "ids": ids}
        return {"y": s["runner"].forward(s["x"], s["ids"], s["w"], s["table"], profile=PROFILES[case["profile"]],
                                         swiglu_limit=SWIGLU_LIMIT)}
    if kind == "route":
        w, ids = ops.route(s["x"], s["gate"], case["topk"], bias=s["bias"], scale=ROUTED_SCALE)
        return {"weights": w, "ids": ids}
    if kind == "dequant":
        return ops.dequant_mxfp4_multi(s["pairs"], tiled=case["tiled"])
    if kind == "quant":
        codes, scale = npu_ops.act_quant(s["x"])
        packed, mx_scale = npu_ops.dynamic_mx_quant(s["x"], case["rule"])
        return {"codes": codes.view(torch.uint8), "scale": scale, "packed": packed, "mx_scale": mx_scale}
    ys = []
    for lay in range(case["layers"]):
        table, _ = s["bank"].acquire_table(lay, s["ids"][lay].cpu().numpy(), case["experts"])
        ys.append(s["runner"].forward(s["x"], s["ids"][lay], s["w"], table, swiglu_limit=SWIGLU_LIMIT))
    return ys


# ---------------------------------------------------------------------------
def _active(tokens, topk, experts):
    """Experts that the Zipf routing of so many tokens reaches (mean of a simulation)."""
    rng = np.random.default_rng(0)
    logp = -ZIPF_S * np.log(np.arange(1, experts + 1))
    n = max(1, min(8, 2048 // tokens))
    got = 0
    for _ in range(n):
        z = logp[None, :] + rng.gumbel(size=(min(tokens, 4096), experts))
        got += np.unique(np.argpartition(-z, topk - 1, axis=1)[:, :topk]).size
    return got / n


def work(case):
    kind = case["kind"]
    D = case["hidden"]
    if kind == "layer":
        T, K, E, I = case["tokens"], case["topk"], case["experts"], case["inter"]
        active = E * (1.0 - (1.0 - K / E) ** T) if case["route"] else _active(T, K, E)
        b = active * 3 * D * I * (0.5 + 1 / 32) + 4 * T * D + 8 * T * K
        f = 6.0 * T * K * D * I
        if case["route"]:
            b += 4 * E * D
            f += 2.0 * T * E * D
        if case["shared"]:
            b += 3 * D * I * (1 + 1 / 32)
            f += 6.0 * T * D * I
        return {"bytes": b, "flops": f}
    if kind == "route":
        T, E = case["tokens"], case["experts"]
        return {"bytes": 4 * E * D + 2 * T * D + 8 * T * case["topk"], "flops": 2.0 * T * E * D}
    if kind == "dequant":
        return {"bytes": 3 * D * case["inter"] * (0.5 + 1 / 32 + 2), "flops": 3 * D * case["inter"]}
    if kind == "quant":
        n = case["tokens"] * D
        return {"bytes": n * (2 + 1 + 4 / 128 + 0.5 + 1 / 32), "flops": 4 * n}
    n = case["layers"] * case["pool"]  # every registered expert is routed to, and copied once
    return {"bytes": n * 3 * D * case["inter"] * (0.5 + 1 / 32) + case["layers"] * 4 * case["tokens"] * D,
            "flops": 6.0 * case["layers"] * case["tokens"] * case["topk"] * D * case["inter"]}


def tolerance(case):
    if case["kind"] in ("dequant", "quant"):
        return "exact"
    if case["kind"] == "route":
        # weights agree to 9e-8 with 64 bits; a near tie of two fp32 scores may order two picks either way
        return {"rel": 2e-3, "max": 0.5, "differ": 1e-3}
    # measured against 64 bits rounded to bf16, at 8 to 16384 tokens: bf16 profile 0.7e-3 to 1.2e-3 and at most
    # 0.04 (a bf16 ulp of a gate/up sum moves an E4M3 code of h now and then); a4w4 up to 4e-5 and 0.018 (its
    # sums are exact, so a code moves rarely, but then by half its value); pure bf16 1.5e-4 and 0.014
    profile = case.get("profile", "bf16")
    return {"rel": {"bf16": 5e-3, "a4w4": 1e-3, "pure": 1e-3}[profile],
            "max": {"bf16": 0.15, "a4w4": 0.08, "pure": 0.06}[profile], "differ": 1e-2}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def _e2m1(nibbles):
    lut = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, 0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0],
                       dtype=torch.float64, device=nibbles.device)
    return lut[nibbles.long()]


def _dequant(codes, scales):
    v = torch.stack((_e2m1(codes & 15), _e2m1(codes >> 4)), -1).flatten(-2)
    return v * torch.exp2(scales.double() - 127).repeat_interleave(32, -1)


def _bf16(x):
    return x.to(torch.bfloat16).double()


def _fp8_blocks(x):
    """(E4M3 codes, block scales) of bf16 values, per 128 columns; the scale is 2^ceil(log2(amax / 448))."""
    v = x.double().unflatten(-1, (-1, 128))
    amax = v.abs().amax(-1, keepdim=True).clamp_min(1e-4)
    s = torch.exp2(torch.ceil(torch.log2(amax / 448.0)))
    return (v / s).clamp(-448, 448).float().to(torch.float8_e4m3fn), s


def _fp8_round_trip(x):
    codes, s = _fp8_blocks(x)
    return (codes.double() * s).flatten(-2)


def _mx_blocks(x, rule):
    """(E2M1 magnitude indexes with the sign in bit 3, block exponents) of bf16 values, per 32 columns."""
    v = x.double().unflatten(-1, (-1, 32))
    amax = v.abs().amax(-1, keepdim=True)
    if rule == "ceil_div6":
        e = torch.ceil(torch.log2(amax.clamp_min(6 * 2.0 ** -126) / 6.0))
    else:
        e = torch.where(amax > 0, torch.floor(torch.log2(amax.clamp_min(2.0 ** -140))) - 2, -127.0).clamp(-127, 127)
    a = (v.abs() * torch.exp2(-e)).clamp_max(6)
    step = torch.exp2(torch.floor(torch.log2(a.clamp_min(1.0))) - 1)  # spacing of the grid at a
    q = torch.round(a / step) * step                                 # ties to even, as the grid's mantissa
    grid = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], dtype=torch.float64, device=x.device)
    mag = torch.searchsorted(grid, q)
    neg = (v * torch.exp2(-e) < 0) if rule == "ceil_div6" else torch.signbit(x).unflatten(-1, (-1, 32))
    return (mag + 8 * neg).to(torch.uint8), e


def _mx_round_trip(x, rule="ocp_floor"):
    nib, e = _mx_blocks(x, rule)
    return (_e2m1(nib) * torch.exp2(e)).flatten(-2)


def _swiglu(gate, up, w):
    gate, up = _bf16(gate).clamp_max(SWIGLU_LIMIT), _bf16(up).clamp(-SWIGLU_LIMIT, SWIGLU_LIMIT)
    return _bf16(gate * torch.sigmoid(gate) * up * w)


def _routed_rows(x, ids, w, experts, weights, profile, expert_of=lambda e: e):
    """sum over each token's picks of its experts' outputs (bf16 GEMM outputs and h, as the layer defines them)."""
    act = {"bf16": _fp8_round_trip, "a4w4": _mx_round_trip, "pure": lambda v: v.double()}[profile]
    xq = act(x)
    y = torch.zeros(x.shape[0], x.shape[1], dtype=torch.float64, device=x.device)
    for e in range(experts):
        tok, k = (ids == e).nonzero(as_tuple=True)
        if tok.numel() == 0:
            continue
        i = expert_of(e)
        w1, w3, w2 = (_dequant(weights[n + "p"][i], weights[n + "s"][i]) for n in ("w1", "w3", "w2"))
        rows = xq[tok]
        h = _swiglu(rows @ w1.T, rows @ w3.T, w[tok, k].double()[:, None])
        y.index_add_(0, tok, _bf16(act(h.to(torch.bfloat16)) @ w2.T))
    return y


def _shared_rows(x, sh):
    def full(n):
        return sh[n].double() * torch.exp2(sh[n + "s"].double() - 127).repeat_interleave(128, 0).repeat_interleave(128, 1)
    xq = _fp8_round_trip(x)
    h = _swiglu(xq @ full("w1").T, xq @ full("w3").T, 1.0)
    return _bf16(_fp8_round_trip(h.to(torch.bfloat16)) @ full("w2").T)


def _route_exact(x, gate, bias, topk):
    scores = torch.sqrt(torch.nn.functional.softplus(x.double() @ gate.double().T, threshold=1e9))
    ids = torch.topk(scores + bias.double(), topk, dim=1).indices
    w = scores.gather(1, ids)
    return w / w.sum(1, keepdim=True) * ROUTED_SCALE, ids.to(torch.int32)


def exact(case, seed):
    kind = case["kind"]
    D = case["hidden"]
    if kind == "layer":
        E, I, T = case["experts"], case["inter"], case["tokens"]
        x = _activations(seed, T, D)
        weights = _experts(seed, E, D, I)
        if not case["route"]:
            ids, w = _routing(seed, T, case["topk"], E)
            return {"y": _routed_rows(x, ids, w, E, weights, case["profile"])}
        w, ids = _route_exact(x, *_gate(seed, E, D), case["topk"])
        y = _routed_rows(x, ids, w, E, weights, case["profile"])
        if case["shared"]:
            y = _bf16(y) + _shared_rows(x, _shared(seed, D, I))
        return {"y": y, "weights": w, "ids": ids}
    if kind == "route":
        w, ids = _route_exact(_activations(seed, case["tokens"], D), *_gate(seed, case["experts"], D), case["topk"])
        return {"weights": w, "ids": ids}
    if kind == "dequant":
        w = _experts(seed, 1, D, case["inter"])
        return [_dequant(w[n + "p"][0], w[n + "s"][0]) for n in ("w1", "w2", "w3")]
    if kind == "quant":
        x = _activations(seed, case["tokens"], D)
        codes, s = _fp8_blocks(x)
        nib, e = _mx_blocks(x, case["rule"])
        nib = nib.flatten(-2)
        return {"codes": codes.flatten(-2).view(torch.uint8), "scale": s[..., 0],
                "packed": nib[..., 0::2] | (nib[..., 1::2] << 4), "mx_scale": (e[..., 0] + 127).to(torch.uint8)}
    x = _activations(seed, case["tokens"], D)
    w = torch.softmax(_normal(_gen(seed, 2), case["tokens"], case["topk"]), 1)
    return [_routed_rows(x, _offload_ids(case, lay).cuda(), w, case["experts"],
                         _experts(seed + 7919 * lay, case["pool"], D, case["inter"]), "bf16", lambda e: e // 2)
            for lay in range(case["layers"])]
