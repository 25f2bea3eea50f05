"""Performance cases of the framework: the calls a Kimi-Linear decoder makes of it.

Every case is one call (or one short chain of calls) through a public entry
point with the operands a serving program holds at that moment: weights and
modules prepared once, activations of one step. Group size 32 is the format of
the reference's own W4A16 checkpoints, group size 128 the format of the
benchmark's configuration; both are run. Shapes are Kimi-Linear's: hidden
2304, 256 routed experts and one shared, intermediate 1024, top-8, attention
projections 2304 -> 4096 and 4096 -> 2304, 32 KDA heads of 128.
"""

from __future__ import annotations

import math

import torch

from local_kimi_amd import kernels, quant
from local_kimi_amd.checkpoint import MoeBanks
from local_kimi_amd.klinear import (KLinearMoE, MoEDecodeGraph, MoELayerTail, RMSNorm, W4A16Linear)

HIDDEN, INTER, EXPERTS, TOP_K, SCALING, EPS = 2304, 1024, 256, 8, 2.446, 1e-5
HEADS, HEAD_DIM = 32, 128
DEV = "cuda"


# ---------------------------------------------------------------------------
# the cases


def listed() -> list[dict]:
    return [
        # one decode token's attention projections, an eager call: launch latency
        {"name": "qkv_decode_1", "op": "qkv", "tokens": 1, "n": 4096, "k": 2304, "group": 32},
        # KDA decode layers of a running batch: recurrent state read and written
        {"name": "kda_decode_16", "op": "kda", "tokens": 16, "heads": 32, "head_dim": 128},
        # one user's decode step of one MoE layer, replayed from its HIP graph
        {"name": "moe_graph_1", "op": "moe_graph", "tokens": 1, "experts": 256, "inter": 1024,
         "group": 128},
        # the post-attention half of a decoder layer on a small serving batch
        {"name": "layer_tail_16", "op": "tail", "tokens": 16, "experts": 256, "inter": 1024,
         "group": 32},
        # a large decode batch with skewed expert popularity
        {"name": "moe_batched_64", "op": "moe", "tokens": 64, "experts": 256, "inter": 1024,
         "group": 128, "routing": "zipf"},
        # a short prompt chunk on MXFP4 experts
        {"name": "mxfp4_moe_200", "op": "mxmoe", "tokens": 200, "experts": 256, "inter": 1024,
         "routing": "normal"},
        # a ragged prompt through one MXFP4 projection with fp16 activations
        {"name": "mxfp4_linear_333", "op": "mxlinear", "tokens": 333, "n": 9216, "k": 2304,
         "dtype": "float16"},
        # o_proj of a ragged prompt at the reference's group size
        {"name": "linear_prefill_1500", "op": "linear", "tokens": 1500, "n": 2304, "k": 4096,
         "group": 32},
        # a prompt's attention projections
        {"name": "qkv_prefill_2048", "op": "qkv", "tokens": 2048, "n": 4096, "k": 2304,
         "group": 128},
        # a ragged prompt through the MoE module at the reference's group size
        {"name": "moe_module_777", "op": "module", "tokens": 777, "experts": 256, "inter": 1024,
         "group": 32},
        # the largest prompt chunk through the MoE block
        {"name": "moe_prefill_2048", "op": "moe", "tokens": 2048, "experts": 256, "inter": 1024,
         "group": 128, "routing": "normal"},
        # quantising an expert-sized stack of weights at load time, and decoding it again
        {"name": "codec_w4a16", "op": "codec", "n": 18432, "k": 2304, "group": 32},
    ]


def _log_int(rng, low: int, high: int) -> int:
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng) -> dict:
    op = rng.choice(["qkv", "qkv", "linear", "linear", "mxlinear", "moe", "moe", "mxmoe", "module",
                     "tail", "moe_graph", "kda", "codec"])
    group = rng.choice([32, 32, 64, 128, 128])
    bank = {"experts": rng.choice([64, 128, 256]), "inter": rng.choice([512, 1024])}
    n, k = rng.choice([(4096, 2304), (2304, 4096), (9216, 2304), (2304, 9216), (576, 2304),
                       (rng.randrange(65, 4096), 256 * rng.randrange(1, 16))])
    if op == "qkv":
        return {"op": op, "tokens": _log_int(rng, 1, 2048), "n": rng.choice([2048, 4096, 1234]),
                "k": 2304, "group": group}
    if op == "linear":
        return {"op": op, "tokens": _log_int(rng, 1, 2048), "n": n, "k": k, "group": group}
    if op == "mxlinear":
        return {"op": op, "tokens": _log_int(rng, 1, 1024), "n": n, "k": k,
                "dtype": rng.choice(["float16", "bfloat16"])}
    if op == "moe":
        return {"op": op, "tokens": _log_int(rng, 1, 2048), **bank, "group": group,
                "routing": rng.choice(["zipf", "normal"])}
    if op == "mxmoe":
        return {"op": op, "tokens": _log_int(rng, 1, 1024), **bank,
                "routing": rng.choice(["zipf", "normal"])}
    if op == "module":
        return {"op": op, "tokens": _log_int(rng, 1, 1024), **bank, "group": group}
    if op == "tail":
        return {"op": op, "tokens": _log_int(rng, 1, 256), **bank, "group": group}
    if op == "moe_graph":
        return {"op": op, "tokens": _log_int(rng, 1, 32), **bank, "group": group}
    if op == "kda":
        return {"op": op, "tokens": _log_int(rng, 1, 64), "heads": rng.choice([16, 32]),
                "head_dim": rng.choice([64, 128])}
    return {"op": op, "n": rng.randrange(256, 32768), "k": rng.choice([1024, 2304, 4096]),
            "group": group}


# ---------------------------------------------------------------------------
# inputs


def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _int4(g, experts: int, n: int, k: int, group: int):
    """Packed codes and scales of N(0, 0.02)-like weights: codes of a group
    spread over [-7, 7] with the group's largest near 7."""
    codes = torch.randn((experts, n, k), generator=g, device=DEV, dtype=torch.float16)
    codes = codes.mul_(2.6).round_().clamp_(-7, 7).to(torch.int8).view(torch.uint8) & 15
    packed = codes[..., 0::2] | (codes[..., 1::2] << 4)
    scales = torch.rand((experts, n, k // group), generator=g, device=DEV).mul_(0.004).add_(0.006)
    return packed, scales.to(torch.bfloat16)


def _fp4(g, experts: int, n: int, k: int):
    """E2M1 codes of rounded normals and block exponents near 2**-7."""
    mag = torch.randn((experts, n, k), generator=g, device=DEV, dtype=torch.float16).mul_(2.5)
    sign = (mag < 0).to(torch.uint8) << 3
    mag = mag.abs_()
    code = (mag >= 0.25).to(torch.uint8)
    for edge in (0.75, 1.25, 1.75, 2.5, 3.5, 5.0):
        code += mag >= edge
    code |= sign
    packed = code[..., 0::2] | (code[..., 1::2] << 4)
    scale = torch.randint(118, 122, (experts, n, k // 32), generator=g, device=DEV).to(torch.uint8)
    return packed, scale


def _hidden(g, tokens: int, width: int, dtype=torch.bfloat16):
    return torch.randn((tokens, width), generator=g, device=DEV).to(dtype)


def _logits(g, tokens: int, experts: int, routing: str):
    if routing == "normal":
        return torch.randn((tokens, experts), generator=g, device=DEV)
    rank = torch.randperm(experts, generator=g, device=DEV).add(1).float()
    u = torch.rand((tokens, experts), generator=g, device=DEV).clamp_(1e-7, 1 - 1e-7)
    return torch.log_softmax(-1.1 * rank.log(), 0)[None, :] - torch.log(-torch.log(u))


def _banks(g, case):
    e, inter = case["experts"] + 1, case["inter"]
    if case["op"] == "mxmoe":
        made = [_fp4(g, e, inter, HIDDEN), _fp4(g, e, inter, HIDDEN), _fp4(g, e, HIDDEN, inter)]
    else:
        made = [_int4(g, e, inter, HIDDEN, case["group"]), _int4(g, e, inter, HIDDEN, case["group"]),
                _int4(g, e, HIDDEN, inter, case["group"])]
    return [t for pair in made for t in pair]


def _inputs(case: dict, seed: int) -> dict:
    """The operands alone, from the seed (shared by prepare and exact)."""
    g, op = _gen(seed), case["op"]
    if op == "qkv":
        x = _hidden(g, case["tokens"], case["k"])
        w = [_int4(g, 1, case["n"], case["k"], case["group"]) for _ in range(3)]
        return {"x": x, "w": [(p[0], s[0]) for p, s in w]}
    if op == "linear":
        p, s = _int4(g, 1, case["n"], case["k"], case["group"])
        return {"x": _hidden(g, case["tokens"], case["k"]), "packed": p[0], "scales": s[0]}
    if op == "mxlinear":
        p, s = _fp4(g, 1, case["n"], case["k"])
        return {"x": _hidden(g, case["tokens"], case["k"], getattr(torch, case["dtype"])),
                "packed": p[0], "scales": s[0]}
    if op in ("moe", "mxmoe"):
        return {"x": _hidden(g, case["tokens"], HIDDEN), "banks": _banks(g, case),
                "logits": _logits(g, case["tokens"], case["experts"], case["routing"])}
    if op in ("module", "moe_graph", "tail"):
        d = {"x": _hidden(g, case["tokens"], HIDDEN), "banks": _banks(g, case),
             "gate": torch.randn((case["experts"], HIDDEN), generator=g, device=DEV)
             .mul_(0.02).to(torch.bfloat16),
             "bias": torch.randn((case["experts"],), generator=g, device=DEV).mul_(0.02)}
        if op == "tail":
            d["delta"] = _hidden(g, case["tokens"], HIDDEN)
            for name in ("ln", "next_ln"):
                d[name] = torch.rand((HIDDEN,), generator=g, device=DEV).add_(0.5).to(torch.bfloat16)
        return d
    if op == "kda":
        b, h, d = case["tokens"], case["heads"], case["head_dim"]
        c = h * d
        r = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
        return {"in": [r(b, 1, c).to(torch.bfloat16) for _ in range(3)],
                "conv": [r(b, c, 4).to(torch.bfloat16) for _ in range(3)],
                "conv_w": [r(c, 1, 4).mul_(0.5).to(torch.bfloat16) for _ in range(3)],
                "raw_decay": r(b, 1, h, d).to(torch.bfloat16), "dt_bias": r(h * d),
                "a_log": torch.rand((1, 1, h, 1), generator=g, device=DEV).mul_(2.0),
                "raw_beta": r(b, 1, h).to(torch.bfloat16), "state": r(b, h, d, d).mul_(0.1)}
    return {"w": torch.randn((case["n"], case["k"]), generator=g, device=DEV).mul_(0.02)
            .to(torch.bfloat16)}


def prepare(case: dict, seed: int):
    d, op = _inputs(case, seed), case["op"]
    d["op"] = op
    if op == "linear":
        d["linear"] = W4A16Linear(quant.W4A16Tensor(
            packed=d["packed"], scales=d["scales"], original_shape=(case["n"], case["k"]),
            group_size=case["group"]))
    elif op in ("module", "moe_graph", "tail"):
        d["moe"] = KLinearMoE(d["gate"], d["bias"], MoeBanks(*d["banks"]), top_k=TOP_K,
                              routed_scaling_factor=SCALING)
        if op == "moe_graph":
            d["graph"] = MoEDecodeGraph(d["moe"], case["tokens"])
        elif op == "tail":
            norms = []
            for name in ("ln", "next_ln"):
                norm = RMSNorm(HIDDEN, EPS, device=DEV, dtype=torch.bfloat16)
                norm.weight.data.copy_(d[name])
                norms.append(norm)
            d["tail"], d["next_norm"] = MoELayerTail(d["moe"], norms[0]), norms[1]
    elif op == "kda":
        d["conv_out"] = [torch.empty_like(t) for t in d["conv"]]
        d["heads"], d["head_dim"] = case["heads"], case["head_dim"]
    elif op == "codec":
        d["group"] = case["group"]
    return d


# ---------------------------------------------------------------------------
# one pass


@torch.no_grad()
def run(s):
    op = s["op"]
    if op == "qkv":
        (qp, qs), (kp, ks), (vp, vs) = s["w"]
        return list(kernels.fused_qkv_w4a16(s["x"], qp, qs, kp, ks, vp, vs))
    if op == "linear":
        return s["linear"](s["x"])
    if op == "mxlinear":
        return kernels.mxfp4_linear(s["x"], s["packed"], s["scales"])
    if op == "moe":
        return list(kernels.w4a16_moe_block(s["x"], s["logits"], None, *s["banks"], TOP_K, SCALING))
    if op == "mxmoe":
        return list(kernels.mxfp4_moe_block(s["x"], s["logits"], None, *s["banks"], TOP_K, SCALING))
    if op == "module":
        return s["moe"](s["x"])
    if op == "moe_graph":
        return s["graph"](s["x"])
    if op == "tail":
        return list(s["tail"](s["x"], s["delta"], s["next_norm"]))
    if op == "kda":
        # a decode loop alternates the two conv-state sets and keeps the state
        out = kernels.kda_decode_layer(
            *s["in"], *s["conv"], *s["conv_w"], s["raw_decay"], s["dt_bias"], s["a_log"],
            s["raw_beta"], s["state"], num_heads=s["heads"], head_dim=s["head_dim"],
            conv_states_out=tuple(s["conv_out"]))
        s["conv"], s["conv_out"] = s["conv_out"], s["conv"]
        return [out, s["state"], *s["conv"]]
    q = quant.quantise(s["w"], group_size=s["group"])
    return [q.packed, q.scales, quant.dequantise(q)]


# ---------------------------------------------------------------------------
# what a pass cannot do without


def _distinct(case: dict) -> float:
    """Expected distinct routed experts of the batch (Monte Carlo for Zipf)."""
    e, t = case["experts"], case["tokens"]
    if case.get("routing") == "zipf":
        g = torch.Generator().manual_seed(0)
        u = torch.rand((8, t, e), generator=g).clamp_(1e-7, 1 - 1e-7)
        score = -1.1 * torch.arange(1, e + 1).float().log() - torch.log(-torch.log(u))
        idx = score.topk(TOP_K, dim=-1).indices
        return sum(len(torch.unique(i)) for i in idx) / 8.0
    return e * (1.0 - (1.0 - TOP_K / e) ** t)


def work(case: dict) -> dict:
    op = case["op"]
    t = case.get("tokens", 0)
    if op == "codec":
        n, k, g = case["n"], case["k"], case["group"]
        packed = n * k / 2 + n * k / g * 2
        return {"bytes": 2 * n * k + packed + packed + 2 * n * k, "flops": 4.0 * n * k}
    if op == "kda":
        h, d = case["heads"], case["head_dim"]
        c = h * d
        state = 2 * 4 * t * c * d
        conv = t * c * 3 * (2 + 2 * 4 * 2) + c * 3 * 8
        gates = t * (c * 2 + h * 2) + c * 4 + h * 4
        return {"bytes": state + conv + gates + t * c * 4, "flops": 8.0 * t * c * d}
    if op in ("qkv", "linear", "mxlinear"):
        n, k = case["n"], case["k"]
        mats = 3 if op == "qkv" else 1
        per = k / 2 + (k / 32 if op == "mxlinear" else 2 * k / case["group"])
        return {"bytes": mats * n * per + 2 * t * k + mats * 2 * t * n, "flops": 2.0 * mats * t * n * k}
    per = 0.5 + (1 / 32 if op == "mxmoe" else 2 / case["group"])
    expert = 3 * HIDDEN * case["inter"]
    nbytes = (_distinct(case) + 1) * expert * per + 4 * t * HIDDEN + 4 * t * case["experts"] + 12 * t * TOP_K
    if op in ("module", "moe_graph", "tail"):
        nbytes += 2 * case["experts"] * HIDDEN - (4 * t * case["experts"] + 12 * t * TOP_K)
        if op == "tail":
            nbytes += 4 * t * HIDDEN + 4 * HIDDEN
        gate = 2.0 * t * case["experts"] * HIDDEN
    else:
        gate = 0.0
    return {"bytes": nbytes, "flops": 2.0 * t * (TOP_K + 1) * expert + gate}


def tolerance(case: dict):
    op = case["op"]
    if op == "codec":
        return "exact"
    if op == "kda":
        # bf16 convolution outputs inside an otherwise fp32 layer
        return {"rel": 8e-3}
    if op == "mxlinear" and case["dtype"] == "float16":
        return {"rel": 1e-3}
    if op in ("qkv", "linear", "mxlinear"):
        return {"rel": 7e-3}  # one rounding to bf16
    # bf16 gate, up, activation and route outputs, and (modules) near-equal experts
    return {"rel": 1.6e-2, "differ": 1e-3}


# ---------------------------------------------------------------------------
# the same in 64 bits


def _dec_int4(packed, scales):
    k = packed.shape[-1] * 2
    q = torch.stack((packed & 15, packed >> 4), dim=-1).reshape(packed.shape[0], k).to(torch.int16)
    q = torch.where(q > 7, q - 16, q).double()
    return (q.reshape(q.shape[0], scales.shape[-1], -1) * scales.double()[..., None]).reshape(q.shape)


def _dec_fp4(packed, scale):
    k = packed.shape[-1] * 2
    c = torch.stack((packed & 15, packed >> 4), dim=-1).reshape(packed.shape[0], k).long()
    grid = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], dtype=torch.float64, device=c.device)
    v = grid[c & 7] * torch.where(c > 7, -1.0, 1.0).double()
    s = torch.exp2(scale.double() - 127.0)
    return (v.reshape(v.shape[0], scale.shape[-1], 32) * s[..., None]).reshape(v.shape)


def _moe64(x, logits, bias, banks, dec):
    score = torch.sigmoid(logits)
    choice = score if bias is None else score + bias.double()
    idx = choice.topk(TOP_K, dim=-1).indices
    w = score.gather(1, idx)
    w = w / (w.sum(-1, keepdim=True) + 1e-20) * SCALING
    experts = logits.shape[1]
    w1p, w1s, w3p, w3s, w2p, w2s = banks
    y = torch.zeros((x.shape[0], HIDDEN), dtype=torch.float64, device=x.device)

    def mlp(e, rows):
        gate, up = rows @ dec(w1p[e], w1s[e]).T, rows @ dec(w3p[e], w3s[e]).T
        return (gate * torch.sigmoid(gate) * up) @ dec(w2p[e], w2s[e]).T

    for e in torch.unique(idx).tolist():
        tok, slot = (idx == e).nonzero(as_tuple=True)
        y.index_add_(0, tok, mlp(e, x[tok]) * w[tok, slot][:, None])
    return y + mlp(experts, x), idx, w


def _rms64(x, weight):
    return weight.double() * x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


@torch.no_grad()
def exact(case: dict, seed: int):
    d, op = _inputs(case, seed), case["op"]
    if op == "qkv":
        return [d["x"].double() @ _dec_int4(p, s).T for p, s in d["w"]]
    if op == "linear":
        return d["x"].double() @ _dec_int4(d["packed"], d["scales"]).T
    if op == "mxlinear":
        return d["x"].double() @ _dec_fp4(d["packed"], d["scales"]).T
    if op in ("moe", "mxmoe"):
        dec = _dec_fp4 if op == "mxmoe" else _dec_int4
        return list(_moe64(d["x"].double(), d["logits"].double(), None, d["banks"], dec))
    if op in ("module", "moe_graph", "tail"):
        x = d["x"].double()
        if op == "tail":
            # the router sees the bf16 rows that the layer itself hands on
            h = (d["x"].float() + d["delta"].float()).to(torch.bfloat16)
            inv = torch.rsqrt(h.float().square().mean(-1, keepdim=True) + EPS)
            x = (d["ln"] * (h.float() * inv).to(torch.bfloat16)).double()
        y = _moe64(x, x @ d["gate"].double().T, d["bias"], d["banks"], _dec_int4)[0]
        if op != "tail":
            return y
        hidden = h.double() + y
        return [hidden, _rms64(hidden, d["next_ln"])]
    if op == "kda":
        b, h, dim = case["tokens"], case["heads"], case["head_dim"]
        conv, outs = [], []
        for x, st, w in zip(d["in"], d["conv"], d["conv_w"]):
            win = torch.cat((st[..., 1:], x[:, 0, :, None]), dim=-1)
            conv.append(win)
            v = (win.double() * w[:, 0, :].double()).sum(-1)
            outs.append((v * torch.sigmoid(v)).reshape(b, h, dim))
        q, k, v = outs
        q = q * torch.rsqrt(q.square().sum(-1, keepdim=True) + 1e-6) * dim ** -0.5
        k = k * torch.rsqrt(k.square().sum(-1, keepdim=True) + 1e-6)
        raw = d["raw_decay"][:, 0].double() + d["dt_bias"].double().reshape(h, dim)
        decay = -torch.exp(d["a_log"].double().reshape(1, h, 1)) * torch.nn.functional.softplus(raw)
        beta = torch.sigmoid(d["raw_beta"][:, 0].double())
        state = d["state"].double() * torch.exp(decay)[..., None]
        delta = (v - (state * k[..., None]).sum(-2)) * beta[..., None]
        state = state + k[..., None] * delta[..., None, :]
        return [(state * q[..., None]).sum(-2), state, *(c.double() for c in conv)]
    w, g = d["w"], case["group"]
    grp = w.float().reshape(w.shape[0], -1, g)
    scale = (grp.abs().amax(-1) / 7.0).to(torch.bfloat16)
    q = (grp / scale.float()[..., None]).round().clamp(-7, 7)
    val = (q.double() * scale.double()[..., None]).reshape(w.shape)
    c = q.to(torch.int8).view(torch.uint8).reshape(w.shape) & 15
    return [c[:, 0::2] | (c[:, 1::2] << 4), scale.double(), val]
