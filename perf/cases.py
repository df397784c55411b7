"""The measured work of this framework: the blocks of a gpt-oss decoder layer, each through the
entry point a program calls.

A case is one call of one block (the MoE experts forward, the experts with their input gradients,
norm + router, attention forward, attention with its gradients, the MXFP4 dequant) at one size.
Shapes are the gpt-oss layers this repository runs everywhere: 2880 wide, 128 experts ("120b") or
32 ("20b"), top-4, 64 query heads over 8 key heads of 64.  Packed weights are uniform MXFP4 codes
with scale bytes in [116, 120] (the range of trained checkpoints: layer outputs of order one),
activations N(0, 1) in bf16, router logits N(0, 1) plus a per-expert bias of deviation 0.5 (experts
are hit unevenly, as in a trained router).
"""

from __future__ import annotations

import math
from types import SimpleNamespace

import torch
from torch import nn

from blockstreamer_amd import attention, gptoss, kernels

DEV = "cuda"
HIDDEN = INTER = 2880
TOP_K = 4
HEADS, KV_HEADS, HEAD_DIM = 64, 8, 64
WINDOW = 128
EPS = 1e-5
ALPHA, LIMIT = 1.702, 7.0
BF16 = torch.bfloat16


def listed():
    return [
        # one token of one chat: four experts' weights, and the launches
        {"name": "experts_decode_t1", "kind": "experts", "experts": 128, "tokens": 1, "layout": "checkpoint"},
        # a serving batch of 64 chats, one token each: most experts hit, a few rows each
        {"name": "experts_decode_t64", "kind": "experts", "experts": 128, "tokens": 64, "layout": "checkpoint"},
        # an ordinary prompt of ragged length: about 31 rows per expert
        {"name": "experts_prompt_t1000", "kind": "experts", "experts": 128, "tokens": 1000, "layout": "checkpoint"},
        # a long prompt, or many packed together
        {"name": "experts_prefill_t8192", "kind": "experts", "experts": 128, "tokens": 8192, "layout": "checkpoint"},
        # a LoRA step on one sequence of 128 tokens: forward that saves, and the input gradients
        {"name": "experts_train_t128", "kind": "experts_train", "experts": 128, "tokens": 128, "layout": "checkpoint"},
        # a LoRA step on 8192 packed tokens
        {"name": "experts_train_t8192", "kind": "experts_train", "experts": 128, "tokens": 8192, "layout": "checkpoint"},
        # what precedes the experts in every layer of that prompt
        {"name": "norm_router_t8192", "kind": "norm_router", "experts": 128, "tokens": 8192},
        # one token each of 8 chats with 4096 cached positions, a full-attention layer
        {"name": "attention_decode_b8_kv4096", "kind": "attention", "batch": 8, "queries": 1, "keys": 4096, "window": 0},
        # a long prompt through a full-attention layer
        {"name": "attention_prefill_t8192", "kind": "attention", "batch": 1, "queries": 8192, "keys": 8192, "window": 0},
        # a training step through a full-attention layer
        {"name": "attention_train_t4096", "kind": "attention_train", "batch": 1, "queries": 4096, "keys": 4096, "window": 0},
        # a training step through a sliding-window layer (every second layer is one)
        {"name": "attention_train_window_t8192", "kind": "attention_train", "batch": 1, "queries": 8192, "keys": 8192,
         "window": WINDOW},
        # the dense weights of one layer's down projections, as a loader materialises them
        {"name": "dequant_down_e128", "kind": "dequant", "experts": 128, "rows": HIDDEN},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["experts", "experts", "experts_train", "norm_router", "attention", "attention",
                       "attention_train", "dequant"])
    if kind in ("experts", "experts_train"):
        return {"kind": kind, "experts": rng.choice([128, 128, 32]),
                "tokens": _log_int(rng, 1 if kind == "experts" else 64, 8192),
                "layout": rng.choice(["checkpoint", "checkpoint", "checkpoint", "kpair"])}
    if kind == "norm_router":
        return {"kind": kind, "experts": rng.choice([128, 32]), "tokens": _log_int(rng, 1, 8192)}
    if kind == "dequant":
        return {"kind": kind, "experts": _log_int(rng, 1, 128), "rows": rng.choice([HIDDEN, 2 * INTER]) // rng.choice([1, 2])}
    window = rng.choice([0, WINDOW])
    if kind == "attention" and rng.random() < 0.5:  # decode: one token per sequence against its cache
        keys = _log_int(rng, 64, 8192)
        return {"kind": kind, "batch": _log_int(rng, 1, min(64, max(1, 64 * 4096 // keys))), "queries": 1, "keys": keys,
                "window": window}
    queries = _log_int(rng, 64, 8192 if kind == "attention" or window else 4096)
    cached = 0 if kind == "attention_train" or rng.random() < 0.7 else _log_int(rng, 1, 8192 - queries + 1)  # chunked prefill
    return {"kind": kind, "batch": _log_int(rng, 1, max(1, min(8, 8192 // queries))), "queries": queries,
            "keys": queries + cached, "window": window}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, dtype=BF16, std=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)


def _packed(g, experts, rows, groups):
    blocks = torch.randint(0, 256, (experts, rows, groups, 16), generator=g, dtype=torch.uint8, device=DEV)
    scales = torch.randint(116, 121, (experts, rows, groups), generator=g, dtype=torch.uint8, device=DEV)
    return blocks, scales


def _expert_inputs(case, seed):
    """Checkpoint-layout tensors of the layer, the hidden states and their routing."""
    g = _gen(seed)
    E, T = case["experts"], case["tokens"]
    t = {}
    t["gate_up_proj_blocks"], t["gate_up_proj_scales"] = _packed(g, E, 2 * INTER, HIDDEN // 32)
    t["down_proj_blocks"], t["down_proj_scales"] = _packed(g, E, HIDDEN, INTER // 32)
    t["gate_up_proj_bias"] = _randn(g, E, 2 * INTER, std=0.01)
    t["down_proj_bias"] = _randn(g, E, HIDDEN, std=0.01)
    hidden = _randn(g, T, HIDDEN)
    logits = torch.randn(T, E, generator=g, device=DEV) + 0.5 * torch.randn(E, generator=g, device=DEV)
    top, idx = logits.topk(TOP_K, dim=-1)
    weights = torch.softmax(top, dim=-1).to(BF16)
    grad = _randn(g, T, HIDDEN, std=0.01)
    return t, hidden, idx, weights, grad


def _norm_inputs(case, seed):
    g = _gen(seed)
    E, T = case["experts"], case["tokens"]
    return (_randn(g, T, HIDDEN, std=4.0), 1.0 + _randn(g, HIDDEN, dtype=torch.float32, std=0.1),
            _randn(g, E, HIDDEN, std=0.02), _randn(g, E, std=0.5))


def _attention_inputs(case, seed):
    """q, k, v as the layer's projections leave them ([B, T, heads, 64] seen as [B, heads, T, 64]), or
    for one-token queries the cache's own [B, heads, T, 64]."""
    g = _gen(seed)
    B, Tq, Tk = case["batch"], case["queries"], case["keys"]

    def kv():
        if Tq == Tk:
            return _randn(g, B, Tk, KV_HEADS, HEAD_DIM).transpose(1, 2)
        return _randn(g, B, KV_HEADS, Tk, HEAD_DIM)

    q = _randn(g, B, Tq, HEADS, HEAD_DIM).transpose(1, 2)
    k, v = kv(), kv()
    sinks = _randn(g, HEADS, dtype=torch.float32)
    grad = _randn(g, B, Tq, HEADS, HEAD_DIM, std=0.01)
    return q, k, v, sinks, grad


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("experts", "experts_train"):
        t, hidden, idx, weights, grad = _expert_inputs(case, seed)
        if case["layout"] == "kpair":
            for name in ("gate_up_proj_blocks", "down_proj_blocks"):
                t[name] = kernels.to_kpair(t[name])
        cfg = SimpleNamespace(num_local_experts=case["experts"], hidden_size=HIDDEN, intermediate_size=INTER,
                              num_experts_per_tok=TOP_K, swiglu_limit=LIMIT)
        layer = gptoss.MXFP4Experts(cfg, BF16)
        for name, value in t.items():
            setattr(layer, name, nn.Parameter(value, requires_grad=False))
        if kind == "experts_train":
            return {"kind": kind, "layer": layer, "hidden": hidden.requires_grad_(True), "idx": idx,
                    "weights": weights.requires_grad_(True), "grad": grad}
        return {"kind": kind, "layer": layer, "hidden": hidden, "idx": idx, "weights": weights}
    if kind == "norm_router":
        hidden, norm_w, router_w, router_b = _norm_inputs(case, seed)
        cfg = SimpleNamespace(num_local_experts=case["experts"], hidden_size=HIDDEN, num_experts_per_tok=TOP_K)
        norm = gptoss.FusedRMSNorm(HIDDEN, EPS, torch.float32, device=DEV)
        router = gptoss.MXFP4TopKRouter(cfg, BF16, device=DEV)
        with torch.no_grad():
            norm.weight.copy_(norm_w)
            router.weight.copy_(router_w)
            router.bias.copy_(router_b)
        return {"kind": kind, "hidden": hidden, "norm": norm, "router": router}
    if kind == "dequant":
        blocks, scales = _packed(_gen(seed), case["experts"], case["rows"], HIDDEN // 32)
        return {"kind": kind, "blocks": blocks, "scales": scales}
    q, k, v, sinks, grad = _attention_inputs(case, seed)
    state = {"kind": kind, "q": q, "k": k, "v": v, "sinks": sinks, "window": case["window"]}
    if kind == "attention_train":
        state["grad"] = grad
        for name in ("q", "k", "v"):
            state[name].requires_grad_(True)
    return state


def run(state):
    kind = state["kind"]
    if kind == "experts":
        with torch.no_grad():
            return state["layer"](state["hidden"], state["idx"], state["weights"])
    if kind == "experts_train":
        out = state["layer"](state["hidden"], state["idx"], state["weights"])
        grad_h, grad_w = torch.autograd.grad(out, (state["hidden"], state["weights"]), state["grad"])
        return {"out": out.detach(), "grad_hidden": grad_h, "grad_weights": grad_w}
    if kind == "norm_router":
        with torch.no_grad():
            normed = state["norm"](state["hidden"])
            logits, scores, idx = state["router"](normed)
        return {"normed": normed, "logits": logits, "scores": scores, "idx": idx}
    if kind == "dequant":
        return kernels.dequantize_mxfp4(state["blocks"], state["scales"], BF16)
    scaling = HEAD_DIM ** -0.5
    if kind == "attention":
        with torch.no_grad():
            return attention.attention(state["q"], state["k"], state["v"], state["sinks"], scaling, True, state["window"])
    out = attention.attention(state["q"], state["k"], state["v"], state["sinks"], scaling, True, state["window"])
    dq, dk, dv = torch.autograd.grad(out, (state["q"], state["k"], state["v"]), state["grad"])
    return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _visible(case):
    """Visible (query, key) pairs of one head."""
    Tq, Tk, w = case["queries"], case["keys"], case["window"]
    n = Tq * (Tk - Tq) + Tq * (Tq + 1) // 2
    if w and w < Tk:
        n = sum(min(w, Tk - Tq + t + 1) for t in range(Tq))
    return n


def work(case):
    kind = case["kind"]
    if kind in ("experts", "experts_train"):
        E, T = case["experts"], case["tokens"]
        hit = E * (1.0 - (1.0 - TOP_K / E) ** T)
        weights = hit * (3 * INTER * HIDDEN * 17 // 32 + 2 * (2 * INTER + HIDDEN))
        rows = T * HIDDEN * 2 * 2 + T * TOP_K * 10
        flops = 6.0 * T * TOP_K * HIDDEN * INTER
        if kind == "experts_train":
            return {"bytes": 2 * weights + 2.5 * rows, "flops": 2 * flops}
        return {"bytes": weights + rows, "flops": flops}
    if kind == "norm_router":
        E, T = case["experts"], case["tokens"]
        return {"bytes": T * HIDDEN * 4 + T * E * 2 + T * TOP_K * 10 + E * HIDDEN * 2, "flops": 2.0 * T * E * HIDDEN}
    if kind == "dequant":
        n = case["experts"] * case["rows"] * HIDDEN
        return {"bytes": n * 17 // 32 + n * 2, "flops": 0}
    B, Tq, Tk = case["batch"], case["queries"], case["keys"]
    seen = min(Tk, case["window"] + Tq - 1) if case["window"] else Tk
    rows = B * HEADS * Tq * HEAD_DIM * 2
    cache = B * KV_HEADS * seen * HEAD_DIM * 2 * 2
    flops = 4.0 * HEAD_DIM * HEADS * B * _visible(case)
    if kind == "attention_train":  # reads q, k, v, grad; writes out, dq, dk, dv
        return {"bytes": 4 * rows + 2 * cache, "flops": 3.5 * flops}
    return {"bytes": 2 * rows + cache, "flops": flops}


def tolerance(case):
    # bf16 operands and outputs: about four times the distance to the 64-bit result measured on an MI355X
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    if kind == "norm_router":  # measured 4.2e-3 (the scores); bf16 logits tie, so the last of the four picks may change
        return {"rel": 1.5e-2, "differ": 0.01}
    if kind == "experts_train":  # measured 3.3e-3 (the hidden states' gradient)
        return {"rel": 1.3e-2}
    if kind == "attention_train":  # measured 2.5e-3
        return {"rel": 1e-2}
    return {"rel": 9e-3}  # measured 2.4e-3 (experts), 2.2e-3 (attention)


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0]


def _dense(blocks, scales, dtype=torch.float64):
    """[R, G, 16] codes and [R, G] exponents as the [R, G*32] weight."""
    lut = torch.tensor(_E2M1, dtype=dtype, device=blocks.device)
    codes = torch.stack((blocks & 15, blocks >> 4), dim=-1).reshape(*blocks.shape[:-1], 32)
    scale = torch.exp2(scales.to(dtype) - 127.0)
    return (lut[codes.long()] * scale[..., None]).reshape(blocks.shape[0], -1)


def _exact_experts(case, seed):
    t, hidden, idx, weights, grad = _expert_inputs(case, seed)
    h, w, go = hidden.double(), weights.double(), grad.double()
    train = case["kind"] == "experts_train"
    out, dh, dw = torch.zeros_like(h), torch.zeros_like(h), torch.zeros_like(w)
    for e in torch.unique(idx).tolist():
        tok, slot = torch.where(idx == e)
        w_gu = _dense(t["gate_up_proj_blocks"][e], t["gate_up_proj_scales"][e])
        w_dn = _dense(t["down_proj_blocks"][e], t["down_proj_scales"][e])
        gu = h[tok] @ w_gu.t() + t["gate_up_proj_bias"][e].double()
        gate, up = gu[:, ::2], gu[:, 1::2]
        g, u = gate.clamp(max=LIMIT), up.clamp(-LIMIT, LIMIT)
        sig = torch.sigmoid(ALPHA * g)
        act = (u + 1) * g * sig
        o = act @ w_dn.t() + t["down_proj_bias"][e].double()
        out.index_add_(0, tok, o * w[tok, slot, None])
        if train:
            dw[tok, slot] = (go[tok] * o).sum(-1)
            d_act = (go[tok] * w[tok, slot, None]) @ w_dn
            d_gu = torch.empty_like(gu)
            d_gu[:, ::2] = d_act * (u + 1) * (sig + ALPHA * g * sig * (1 - sig)) * (gate <= LIMIT)
            d_gu[:, 1::2] = d_act * g * sig * (up.abs() <= LIMIT)
            dh.index_add_(0, tok, d_gu @ w_gu)
    return {"out": out, "grad_hidden": dh, "grad_weights": dw} if train else out


def _exact_norm_router(case, seed):
    hidden, norm_w, router_w, router_b = _norm_inputs(case, seed)
    x = hidden.double()
    normed = norm_w.double() * x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    logits = normed @ router_w.double().t() + router_b.double()
    return {"normed": normed, "logits": logits, "scores": torch.softmax(logits.topk(TOP_K, dim=-1)[0], dim=-1), "idx": None}


def _exact_attention(case, seed):
    q, k, v, sinks, grad = _attention_inputs(case, seed)
    B, Tq, Tk = case["batch"], case["queries"], case["keys"]
    train = case["kind"] == "attention_train"
    G = HEADS // KV_HEADS
    scaling = HEAD_DIM ** -0.5
    pos = torch.arange(Tq, device=DEV)[:, None] + (Tk - Tq)
    key = torch.arange(Tk, device=DEV)[None, :]
    hide = key > pos
    if case["window"]:
        hide = hide | (key <= pos - case["window"])
    out = torch.empty(B, Tq, HEADS, HEAD_DIM, dtype=torch.float64, device=DEV)
    dq = torch.empty(B, HEADS, Tq, HEAD_DIM, dtype=torch.float64, device=DEV)
    dk = torch.zeros(B, KV_HEADS, Tk, HEAD_DIM, dtype=torch.float64, device=DEV)
    dv = torch.zeros_like(dk)
    for b in range(B):
        for h in range(HEADS):
            qh, kh, vh = q[b, h].double(), k[b, h // G].double(), v[b, h // G].double()
            s = (qh @ kh.t() * scaling).masked_fill_(hide, -math.inf)
            sink = sinks[h].double()
            m = torch.maximum(s.max(-1, keepdim=True)[0], sink)
            p = torch.exp(s - m)
            p = p / (p.sum(-1, keepdim=True) + torch.exp(sink - m))
            o = p @ vh
            out[b, :, h] = o
            if train:
                go = grad[b, :, h].double()
                ds = p * (go @ vh.t() - (go * o).sum(-1, keepdim=True)) * scaling
                dq[b, h] = ds @ kh
                dk[b, h // G] += ds.t() @ qh
                dv[b, h // G] += p.t() @ go
    return {"out": out, "dq": dq, "dk": dk, "dv": dv} if train else out


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind in ("experts", "experts_train"):
            return _exact_experts(case, seed)
        if kind == "norm_router":
            return _exact_norm_router(case, seed)
        if kind == "dequant":
            blocks, scales = _packed(_gen(seed), case["experts"], case["rows"], HIDDEN // 32)
            # float32 holds every product of a code and a power of two in this range exactly
            return torch.stack([_dense(b, s, torch.float32).t() for b, s in zip(blocks, scales)])
        return _exact_attention(case, seed)
