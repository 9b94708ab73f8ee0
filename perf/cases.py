"""Measured workloads of the MI355X MoE expert path, through its public entry
points.

A case is a dict of plain values; ``kind`` says which entry points one pass
goes through:

  layer    inference of one MoE layer: ``ops.router_route`` then
           ``ops.experts_forward`` (router, dispatch, experts, combine)
  graph    the same layer captured once as ``graph.MoELayerGraph`` and
           replayed on a new input: what a decode loop keeps
  experts  inference through the converted module ``HipGroupedExperts`` on
           routing that the caller already has (an expert shard)
  fp8      ``functional.moe_experts_forward_fp8`` on pre-quantised weights
  train    ``functional.router`` and the converted module, forward and
           backward, optionally with the always-on shared expert
  regroup  the dispatcher's expert-parallel ``_permute`` and ``_unpermute``

Shapes are the model shapes that this repository is configured, tested and
benchmarked with.  Inputs are x ~ N(0, 1) and weights ~ N(0, 0.02); a router
over N(0, 1) tokens loads the experts nearly evenly, and an expert shard gets
a Zipf(1.2) load with some experts empty.
"""
from __future__ import annotations

import importlib
import math

import numpy as np
import torch

_PKG = "torchtitan-ascend_amd"
_DEV = "cuda"
_BF16 = torch.bfloat16

# D, H, experts, top-k, score function, renormalise, scores before the experts
_SHAPES = {
    # Llama4 debug model: the small model of development runs
    "debug": dict(D=256, H=512, E=8, K=1, score="sigmoid", norm=False, before=True),
    # Qwen3-30B-A3B: many small experts, top-8
    "qwen3": dict(D=2048, H=768, E=128, K=8, score="softmax", norm=True, before=False),
    # Llama4-Scout: few large experts, top-1, shared expert
    "scout": dict(D=5120, H=8192, E=16, K=1, score="sigmoid", norm=False, before=True),
    # DeepSeek-V3: one GPU's 32 experts of 256, rows already sent to it
    "shard": dict(D=7168, H=2048, E=32, K=1, score="given", norm=False, before=False),
}


def _case(kind, shape, T, **options):
    c = dict(kind=kind, T=T, limit=0.0, shared=False, param="bf16", zipf=0.0, empty=0, ranks=1)
    c.update(_SHAPES[shape])
    c.update(options)
    return c


def listed():
    cases = [
        # one sequence decoding, eager: eight experts' weights, launches and host
        ("qwen3_decode_1", _case("layer", "qwen3", 1)),
        # a decode batch in a serving loop, replayed as a graph
        ("qwen3_decode_32", _case("graph", "qwen3", 32)),
        # a short ragged prefill: every expert hit, few rows each
        ("qwen3_prefill_1003", _case("layer", "qwen3", 1003)),
        # a full prefill batch: the headline layer forward
        ("qwen3_prefill_8192", _case("layer", "qwen3", 8192)),
        # the debug model's layer: small matrices, eager
        ("debug_layer_2048", _case("layer", "debug", 2048)),
        # an expert shard while its ranks decode: Zipf load, 200 rows in all
        ("shard_decode_200", _case("experts", "shard", 200, zipf=1.2, empty=4)),
        # an expert shard while its ranks prefill
        ("shard_prefill_32768", _case("experts", "shard", 32768, zipf=1.2, empty=4)),
        # the same two with e4m3 weights and activations
        ("shard_fp8_decode_200", _case("fp8", "shard", 200, zipf=1.2, empty=4)),
        ("shard_fp8_prefill_32768", _case("fp8", "shard", 32768, zipf=1.2, empty=4)),
        # a training micro-batch, fp32 Parameters (what the modules hold by default)
        ("qwen3_train_4096", _case("train", "qwen3", 4096, param="fp32")),
        # the largest: a training step of the large top-1 layer and its shared expert
        ("scout_train_8192", _case("train", "scout", 8192, shared=True)),
        # rows of 8 ranks regrouped expert-major and back
        ("regroup_8x32", _case("regroup", "shard", 32768, zipf=1.2, empty=4, ranks=8)),
    ]
    return [dict(c, name=n) for n, c in cases]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "graph", "experts", "fp8", "train", "train", "regroup"])
    limit = rng.choice([0.0, 0.0, 7.0])
    if kind == "layer":
        shape = rng.choice(["qwen3", "qwen3", "debug"])
        c = _case(kind, shape, _log_int(rng, 1, 8192), limit=limit)
        if shape == "qwen3":
            c.update(K=rng.choice([8, 8, 4, 2]), E=rng.choice([128, 128, 64]))
        return c
    if kind == "graph":
        shape = rng.choice(["qwen3", "qwen3", "debug"])
        return _case(kind, shape, _log_int(rng, 1, 512), limit=limit)
    if kind in ("experts", "fp8"):
        empty = rng.choice([0, 4, 9])
        return _case(kind, "shard", _log_int(rng, 32, 32768), zipf=rng.choice([0.0, 0.7, 1.2]), empty=empty,
                     limit=limit, before=rng.random() < 0.25)
    if kind == "train":
        shape = rng.choice(["qwen3", "debug", "scout"])
        return _case(kind, shape, _log_int(rng, 64, 4096 if shape == "qwen3" else 8192), limit=limit,
                     param=rng.choice(["bf16", "fp32"]) if shape != "scout" else "bf16",
                     shared=rng.random() < 0.5)
    return _case(kind, "shard", _log_int(rng, 64, 32768), zipf=rng.choice([0.0, 1.2]), empty=rng.choice([0, 4]),
                 ranks=rng.choice([2, 4, 8]))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _mod(name=None):
    return importlib.import_module(_PKG if name is None else f"{_PKG}.{name}")


def _normal(gen, *shape, std=1.0):
    return torch.randn(*shape, generator=gen, device=_DEV, dtype=_BF16).mul_(std)


def _counts(case, rows=None):
    """Rows per expert of a shard: Zipf over the non-empty experts, the same
    for every seed, on a fixed spread of the experts."""
    rows = case["T"] * case["K"] if rows is None else rows
    E, n = case["E"], case["E"] - case["empty"]
    w = np.arange(1, n + 1, dtype=np.float64) ** -case["zipf"]
    c = np.floor(rows * w / w.sum()).astype(np.int64)
    c[0] += rows - c.sum()
    counts = np.zeros(E, np.int64)
    counts[np.random.default_rng(E).permutation(E)[:n]] = c
    return counts


def _labels(case, seed):
    lab = np.repeat(np.arange(case["E"]), _counts(case))
    return torch.from_numpy(np.random.default_rng(seed).permutation(lab)).to(_DEV).view(case["T"], case["K"])


def _module(case, dtype):
    """The expert module as the two converters build it."""
    pkg, P = _mod(), _mod("protocol")
    mc = P.ModelConfig()
    mc.moe = P.GroupedExperts.Config(
        dim=case["D"], hidden_dim=case["H"], num_experts=case["E"],
        token_dispatcher=P.AllToAllTokenDispatcher.Config(num_experts=case["E"], top_k=case["K"],
                                                          score_before_experts=case["before"]))
    pkg.HipGroupedExpertsConverter(pkg.HipGroupedExpertsConverter.Config(swiglu_limit=_limit(case))).convert(mc)
    pkg.HipTokenDispatcherConverter(pkg.HipTokenDispatcherConverter.Config()).convert(mc)
    with torch.device(_DEV):
        return mc.moe.build().to(dtype)


def _limit(case):
    return case["limit"] if case["limit"] > 0 else None


def prepare(case, seed):
    gen = torch.Generator(device=_DEV)
    gen.manual_seed(seed)
    kind, T, D, H, E = (case[k] for k in ("kind", "T", "D", "H", "E"))
    s = dict(case=case)
    if kind == "regroup":
        counts = _counts(case)
        split = np.random.default_rng(seed)
        group = np.stack([split.multinomial(int(n), np.full(case["ranks"], 1.0 / case["ranks"])) for n in counts])
        s["counts"] = torch.from_numpy(np.ascontiguousarray(group.T).reshape(-1)).to(_DEV)
        s["rows"] = _normal(gen, T, D)
        td = _mod("token_dispatcher").HipTokenDispatcher
        s["dispatcher"] = td(td.Config(num_experts=E, top_k=1, score_before_experts=False))
        return s
    s["x"] = _normal(gen, T, D)
    w13 = _normal(gen, E, 2 * H, D, std=0.02)
    w2 = _normal(gen, E, D, H, std=0.02)
    if case["score"] == "given":
        s["scores"] = torch.rand(T, case["K"], generator=gen, device=_DEV)
        s["idx"] = _labels(case, seed)
    else:
        s["w_router"] = _normal(gen, E, D, std=0.02)
    if kind == "fp8":
        # a checkpoint's quantised weights
        ops = _mod("ops")
        s["w13"], s["s13"] = ops.quantize_fp8_blocks(w13)
        s["w2"], s["s2"] = ops.quantize_fp8_blocks(w2)
        return s
    if kind in ("experts", "train"):
        m = _module(case, torch.float32 if case["param"] == "fp32" else _BF16)
        with torch.no_grad():
            m.w13.copy_(w13)
            m.w2.copy_(w2)
        s["module"] = m
    else:
        s["w13"], s["w2"] = w13, w2
    if kind == "graph":
        s["graph"] = _mod("graph").MoELayerGraph(s["x"], s["w_router"], w13, w2, case["K"], case["score"],
                                                 case["norm"], case["before"], swiglu_limit=_limit(case))
    if kind == "train":
        s["dout"] = _normal(gen, T, D)
        s["x"].requires_grad_(True)
        dt = torch.float32 if case["param"] == "fp32" else _BF16
        s["w_router"] = s["w_router"].to(dt).requires_grad_(True)
        if case["shared"]:
            s["w13_shared"] = _normal(gen, 2 * H, D, std=0.02).to(dt).requires_grad_(True)
            s["w2_shared"] = _normal(gen, D, H, std=0.02).to(dt).requires_grad_(True)
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind, T, D, K = case["kind"], case["T"], case["D"], case["K"]
    if kind == "train":
        return _train_step(state)
    with torch.no_grad():
        if kind == "layer":
            ops = _mod("ops")
            scores, idx, r = ops.router_route(state["x"], state["w_router"], K, case["score"], case["norm"],
                                              with_inverse=False)
            out = ops.experts_forward(state["x"], r, state["w13"], state["w2"], K, case["before"], _limit(case))
            return out, scores, idx
        if kind == "graph":
            return state["graph"](state["x"])
        if kind == "experts":
            return state["module"](state["x"].view(1, T, D), state["scores"], state["idx"])
        if kind == "fp8":
            return _mod("functional").moe_experts_forward_fp8(
                state["x"], state["scores"], state["idx"], state["w13"], state["s13"], state["w2"], state["s2"],
                case["E"], case["before"], _limit(case))
        shape, permuted, order, counts = state["dispatcher"]._permute(
            state["rows"], state["counts"], case["ranks"], case["E"])
        return permuted, order, counts, state["dispatcher"]._unpermute(permuted, shape, order)


def _train_step(state):
    case, F, m = state["case"], _mod("functional"), state["module"]
    leaves = [state["x"], state["w_router"], m.w13, m.w2]
    if case["shared"]:
        leaves += [state["w13_shared"], state["w2_shared"]]
    for p in leaves:
        p.grad = None
    x, T, D = state["x"], case["T"], case["D"]
    scores, idx = F.router(x, state["w_router"], case["K"], case["score"], case["norm"])
    out = m(x.view(1, T, D), scores, idx).view(T, D)
    if case["shared"]:
        out = F.shared_expert_combine(out, x, state["w13_shared"], state["w2_shared"], None, _limit(case))
    out.backward(state["dout"])
    return [out.detach()] + [p.grad for p in leaves]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _active(case):
    """Experts that get a row: exact for a shard, expected for a router."""
    if case["score"] == "given":
        return int((_counts(case) > 0).sum())
    E, K = case["E"], case["K"]
    return E * (1.0 - (1.0 - K / E) ** case["T"])


def work(case):
    kind, T, D, H, E, K = (case[k] for k in ("kind", "T", "D", "H", "E", "K"))
    rows = T * K
    if kind == "regroup":
        # rows in, permuted out, and back; labels' order
        return {"bytes": 2 * (2 * T * D * 2) + 4 * T, "flops": 0}
    weights = _active(case) * 3 * H * D
    flops = 6 * rows * D * H
    if kind == "fp8":
        return {"bytes": weights * (1 + 4 / 16384) + 2 * T * D * 2 + 12 * rows, "flops": flops}
    routed = 2 * T * D * 2 + 12 * rows  # x in, out written, scores and ids
    gate = 0 if case["score"] == "given" else 1
    if kind != "train":
        return {"bytes": weights * 2 + routed + gate * E * D * 2, "flops": flops + gate * 2 * T * D * E}
    size = 4 if case["param"] == "fp32" else 2
    sh = 1 if case["shared"] else 0
    # weights read, their gradients written (whole tensors), x, out, dout, dx
    every = (E * 3 * H * D + E * D + sh * 3 * H * D) * size
    return {"bytes": (_active(case) + sh) * 3 * H * D * size + every + 4 * T * D * 2 + 12 * rows,
            "flops": 3 * (flops + sh * 6 * T * D * H + 2 * T * D * E)}


def tolerance(case):
    """About four times the measured distance from ``exact``: 3e-3 to 4.3e-3
    for bf16 outputs and gradients (the bf16 rounding of the pre-activation,
    the activation and the result; 0.5 % for one token's pick that falls on
    the other side of a logit tie), 1.5e-2 for fp8 (the bf16 rounding of the
    activations before their e4m3 codes)."""
    kind = case["kind"]
    if kind == "regroup":
        return "exact"
    if kind == "fp8":
        return {"rel": 4e-2}
    if kind == "train":
        return {"rel": 2e-2}
    return {"rel": 1.6e-2, "differ": 2e-3}


# ---------------------------------------------------------------------------
# The same in 64 bits, plain torch
# ---------------------------------------------------------------------------
def _router64(x, w_router, case):
    """The gate Linear's output is bf16 by the router's contract, so the 64-bit
    logits are rounded to it once; everything after is 64 bits.  Ties go to
    the lower expert."""
    logits = x @ w_router.t()
    logits = logits + (logits.detach().to(_BF16).double() - logits.detach())
    p = torch.softmax(logits, 1) if case["score"] == "softmax" else torch.sigmoid(logits)
    idx = torch.sort(p.detach(), dim=1, descending=True, stable=True).indices[:, :case["K"]].contiguous()
    scores = p.gather(1, idx)
    if case["norm"]:
        scores = scores / (scores.sum(1, keepdim=True) + 1e-20)
    return scores, idx


def _ffn64(x, w13, w2, limit):
    gate, up = (x @ w13.t()).chunk(2, dim=1)
    if limit is not None:
        gate, up = gate.clamp(max=limit), up.clamp(-limit, limit)
    return (torch.nn.functional.silu(gate) * up) @ w2.t()


def _experts64(x, scores, idx, w13, w2, case, ffn=_ffn64):
    out = torch.zeros_like(x)
    for e in range(case["E"]):
        t, k = (idx == e).nonzero(as_tuple=True)
        if t.numel():
            s = scores[t, k].unsqueeze(1)
            xe = x[t] * s if case["before"] else x[t]
            y = ffn(xe, w13(e), w2(e), _limit(case))
            out = out.index_add(0, t, y if case["before"] else y * s)
    return out


def _codes64(a):
    """e4m3 codes of each row's 128-channel groups (scale absmax / 448), dequantised."""
    g = a.reshape(a.shape[0], -1, 128)
    scale = g.abs().amax(2, keepdim=True).clamp(min=1e-30) / 448.0
    return ((g / scale).float().to(torch.float8_e4m3fn).double() * scale).reshape(a.shape)


def _ffn64_fp8(x, w13, w2, limit):
    gate, up = (_codes64(x) @ w13.t()).chunk(2, dim=1)
    if limit is not None:
        gate, up = gate.clamp(max=limit), up.clamp(-limit, limit)
    return _codes64(torch.nn.functional.silu(gate) * up) @ w2.t()


def _blocks64(q, scale):
    N, K = q.shape
    w = q.view(torch.float8_e4m3fn).double().view(N // 128, 128, K // 128, 128)
    return (w * scale.double()[:, None, :, None]).reshape(N, K)


def exact(case, seed):
    s = prepare(case, seed)
    kind, T = case["kind"], case["T"]
    if kind == "regroup":
        labels = torch.arange(case["E"], device=_DEV).repeat(case["ranks"]).repeat_interleave(s["counts"])
        order = torch.argsort(labels, stable=True)  # int32 below, as the dispatcher returns it
        counts = s["counts"].view(case["ranks"], -1).sum(0)
        return s["rows"][order], order.int(), counts, s["rows"]
    if kind == "train":
        return _train64(s)
    with torch.no_grad():
        x = s["x"].double()
        if case["score"] == "given":
            scores, idx = s["scores"].double(), s["idx"]
        else:
            scores, idx = _router64(x, s["w_router"].double(), case)
        if kind == "fp8":
            out = _experts64(x, scores, idx, lambda e: _blocks64(s["w13"][e], s["s13"][e]),
                             lambda e: _blocks64(s["w2"][e], s["s2"][e]), case, _ffn64_fp8)
            return out
        w13, w2 = (s["module"].w13, s["module"].w2) if kind == "experts" else (s["w13"], s["w2"])
        out = _experts64(x, scores, idx, lambda e: w13[e].double(), lambda e: w2[e].double(), case)
        if kind == "layer":
            return out, scores, idx
        return out if kind == "graph" else out.view(1, T, -1)


def _train64(s):
    case, m = s["case"], s["module"]
    E = case["E"]

    def leaf(t):
        return t.detach().double().requires_grad_(True)

    x, wr = leaf(s["x"]), leaf(s["w_router"].to(_BF16))
    w13 = [leaf(m.w13[e].to(_BF16)) for e in range(E)]
    w2 = [leaf(m.w2[e].to(_BF16)) for e in range(E)]
    scores, idx = _router64(x, wr, case)
    out = _experts64(x, scores, idx, w13.__getitem__, w2.__getitem__, case)
    shared = []
    if case["shared"]:
        shared = [leaf(s["w13_shared"].to(_BF16)), leaf(s["w2_shared"].to(_BF16))]
        out = out + _ffn64(x, shared[0], shared[1], _limit(case))
    out.backward(s["dout"].double())

    def stacked(ws):
        return torch.stack([torch.zeros_like(w) if w.grad is None else w.grad for w in ws])

    return [out.detach(), x.grad, wr.grad, stacked(w13), stacked(w2)] + [w.grad for w in shared]
