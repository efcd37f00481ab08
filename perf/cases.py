"""Performance cases of the MoE layer: the calls that a program serving a mixture-of-experts
model makes, through ``HybridMoE`` and ``FusedMoEBlock``.

A case is one pass over ``layers`` MoE layers (each with its own weights and input, as in a
model, where attention stands between them) on ``tokens`` tokens:

  model   the layer's architecture and weight format: Qwen3-30B-A3B (int4 group-128, int8 per
          channel or bf16 experts), Mixtral-8x7B (int4), Qwen1.5-MoE (int8 with its shared expert)
  call    "layer": HybridMoE.forward(hidden_states, router_logits); "block": FusedMoEBlock.forward
          (RMSNorm, router, experts, residual) on hidden states
  replay  True: the pass was captured in a HIP graph and is replayed, as a serving loop decodes;
          False: eager calls
  zipf    exponent of the router's popularity bias -zipf * ln(expert + 1); 0 = even routing
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-ktrans_amd"))

from nano_ktrans_amd import GPTQLinearWeight, HybridMoE, PackedSparseExpertMLP, SparseExpertMLP  # noqa: E402
from nano_ktrans_amd.layers.moe_block import FusedMoEBlock  # noqa: E402

QWEN3 = dict(H=2048, E=128, k=8, I=768, Is=0, softmax=True, renorm=True)
MODELS = {
    "qwen3_int4": dict(QWEN3, bits=4),
    "qwen3_int8": dict(QWEN3, bits=8),
    "qwen3_bf16": dict(QWEN3, bits=16),
    "mixtral_int4": dict(H=4096, E=8, k=2, I=14336, Is=0, softmax=False, renorm=True, bits=4),
    "qwen15_int8": dict(H=2048, E=60, k=4, I=1408, Is=5632, softmax=True, renorm=False, bits=8),
}
STD = 0.02        # of router and expert weights
EPS = 1e-6        # of the block's RMSNorm


def _case(name, model, tokens, *, layers=1, call="layer", replay=False, zipf=0.0):
    c = {"model": model, "tokens": tokens, "layers": layers, "call": call, "replay": replay, "zipf": zipf}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one token through one layer without a graph: the call's own latency, host side included
        _case("q3_int4_t1_eager", "qwen3_int4", 1),
        # single-stream decoding: a few experts per layer, launch latency against little traffic
        _case("q3_int4_t1", "qwen3_int4", 1, layers=6, replay=True),
        # batched decoding, the ordinary serving step: most experts' weights read once
        _case("q3_int4_t16", "qwen3_int4", 16, layers=3, replay=True),
        # a decoder layer's MoE half (norm, router, experts, residual) for a large decode batch
        _case("q3_int4_block_t48", "qwen3_int4", 48, layers=3, call="block", replay=True),
        # decoding with a shared expert, int8, an odd batch
        _case("q15_int8_t13", "qwen15_int8", 13, layers=3, replay=True),
        # few large experts, a small odd batch
        _case("mixtral_int4_t3", "mixtral_int4", 3, replay=True),
        # a short prompt, or the ragged end of a chunked prefill
        _case("q3_int4_t203", "qwen3_int4", 203),
        # a default 512-token prefill chunk under skewed routing
        _case("q3_int8_t512_zipf", "qwen3_int8", 512, zipf=1.1),
        # prompt batches: long prefill of each model and weight format
        _case("q3_int4_t2048", "qwen3_int4", 2048),
        _case("q3_int8_t4096_zipf", "qwen3_int8", 4096, zipf=1.1),
        _case("q3_bf16_t1000", "qwen3_bf16", 1000),
        _case("mixtral_int4_t2048", "mixtral_int4", 2048),
    ]


def _log_int(rng, lo, hi):
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["eager", "decode", "decode", "prefill", "prefill", "prefill"])
    if kind == "eager":
        return _case("", rng.choice(["qwen3_int4", "qwen3_int8", "qwen15_int8"]), _log_int(rng, 1, 16))
    if kind == "decode":
        model = rng.choice(["qwen3_int4", "qwen3_int8", "qwen3_bf16", "mixtral_int4", "qwen15_int8"])
        layers = 1 if model == "mixtral_int4" else rng.randint(2, 3)
        call = "layer" if model == "qwen15_int8" else rng.choice(["layer", "layer", "block"])
        return _case("", model, _log_int(rng, 1, 64), layers=layers, call=call, replay=True)
    model = rng.choice(["qwen3_int4", "qwen3_int8", "qwen3_bf16", "mixtral_int4", "qwen15_int8"])
    tokens = _log_int(rng, 65, 2048 if model == "mixtral_int4" else 4096)
    return _case("", model, tokens, zipf=rng.choice([0.0, 1.1]))


# ------------------------------------------------------------------ inputs
def _quantized(g, experts, n, k, bits):
    """Symmetric codes of N(0, STD) weights [experts, n, k], packed into int32 words as the
    checkpoints store them, and their scales [experts, n, groups] (bf16 values): int4 in groups
    of 128 inputs, int8 with one scale per row."""
    group, top = (128, 7) if bits == 4 else (k, 127)
    per = 32 // bits
    words = torch.empty(experts, n, k // per, dtype=torch.int32, device="cuda")
    scales = torch.empty(experts, n, k // group, dtype=torch.float32, device="cuda")
    step = max(1, (1 << 28) // (n * k))
    for e in range(0, experts, step):
        w = torch.randn(min(step, experts - e), n, k // group, group, generator=g, device="cuda").mul_(STD)
        s = (w.abs().amax(dim=3) / top).to(torch.bfloat16).to(torch.float32)
        q = w.div_(s.unsqueeze(3)).round_().clamp_(-top - 1, top).add_(top + 1).to(torch.int32)
        q = q.view(q.shape[0], n, k // per, per)
        packed = q[..., 0].clone()
        for j in range(1, per):
            packed |= q[..., j] << (bits * j)
        words[e:e + step] = packed
        scales[e:e + step] = s
    return words, scales


def _weights(m, g):
    """One layer's checkpoint: {"gate_up", "down"[, "shared_gate_up", "shared_down", "shared_gate"], "router", "norm"};
    a projection is (words, scales) or a bf16 tensor, experts first, gate rows before up rows."""
    def proj(experts, n, k):
        if m["bits"] == 16:
            return torch.empty(experts, n, k, dtype=torch.bfloat16, device="cuda").normal_(0, STD, generator=g)
        return _quantized(g, experts, n, k, m["bits"])

    w = {"gate_up": proj(m["E"], 2 * m["I"], m["H"]), "down": proj(m["E"], m["H"], m["I"])}
    if m["Is"]:
        w["shared_gate_up"] = proj(1, 2 * m["Is"], m["H"])
        w["shared_down"] = proj(1, m["H"], m["Is"])
        w["shared_gate"] = (torch.randn(1, m["H"], generator=g, device="cuda") * STD).to(torch.bfloat16)
    w["router"] = (torch.randn(m["E"], m["H"], generator=g, device="cuda") * STD).to(torch.bfloat16)
    w["norm"] = (1 + 0.1 * torch.randn(m["H"], generator=g, device="cuda")).to(torch.bfloat16)
    return w


def _inputs(case, m, w, g):
    x = torch.randn(case["tokens"], m["H"], generator=g, device="cuda").to(torch.bfloat16)
    logits = x.float() @ w["router"].float().T
    logits -= case["zipf"] * torch.log(torch.arange(m["E"], device="cuda") + 1.0)
    return x, logits.to(torch.bfloat16)


def _seeded(case, seed, layer):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 64 + layer)
    return g


def _gptq(q, expert, rows, bits):
    words, scales = q[0][expert, rows], q[1][expert, rows]
    group = 128 if bits == 4 else words.shape[1] * 4
    return GPTQLinearWeight(qweight=words, scales=scales, zero_points=None, group_size=group, bits=bits, sym=True,
                            linear_prefix="")


def _dense(q, expert):
    """float64 weight of one expert's projection."""
    if isinstance(q, torch.Tensor):
        return q[expert].double()
    words, scales = q[0][expert], q[1][expert].double()
    bits = 4 if scales.shape[1] > 1 else 8
    codes = torch.stack([(words >> (bits * j)) & ((1 << bits) - 1) for j in range(32 // bits)], dim=-1)
    codes = codes.reshape(words.shape[0], scales.shape[1], -1).double() - (1 << (bits - 1))
    return (codes * scales.unsqueeze(2)).reshape(words.shape[0], -1)


class _RMSNorm(torch.nn.Module):
    def __init__(self, weight):
        super().__init__()
        self.weight = torch.nn.Parameter(weight, requires_grad=False)
        self.eps = EPS


def _linear(weight):
    with torch.device("meta"):
        lin = torch.nn.Linear(weight.shape[1], weight.shape[0], bias=False)
    lin.weight = torch.nn.Parameter(weight, requires_grad=False)
    return lin


def _module(case, m, w):
    gate, up = slice(0, m["I"]), slice(m["I"], 2 * m["I"])
    experts, quantized, shared = {}, {}, {}
    if m["bits"] == 16:
        for e in range(m["E"]):
            with torch.device("meta"):
                mlp = PackedSparseExpertMLP(m["H"], m["I"])
            mlp.gate_up_proj = torch.nn.Parameter(w["gate_up"][e], requires_grad=False)
            mlp.down_proj = _linear(w["down"][e])
            experts[str(e)] = mlp
    else:
        for e in range(m["E"]):
            quantized[e] = {"gate": _gptq(w["gate_up"], e, gate, m["bits"]),
                            "up": _gptq(w["gate_up"], e, up, m["bits"]),
                            "down": _gptq(w["down"], e, slice(None), m["bits"])}
    if m["Is"]:
        # the dense shared expert of the checkpoint, quantized at ingest like the routed ones were
        gu, down = _dense(w["shared_gate_up"], 0).float(), _dense(w["shared_down"], 0).float()
        with torch.device("meta"):
            mlp = SparseExpertMLP(m["H"], m["Is"])
        mlp.w1, mlp.w3, mlp.w2 = _linear(gu[:m["Is"]]), _linear(gu[m["Is"]:]), _linear(down)
        shared = {"shared_expert": mlp, "shared_expert_gate": _linear(w["shared_gate"]),
                  "quantization": "int8_per_channel"}
    moe = HybridMoE(
        num_experts=m["E"], top_k=m["k"], hidden_size=m["H"], moe_intermediate_size=m["I"],
        gpu_experts=torch.nn.ModuleDict(experts), gpu_experts_mask=torch.ones(m["E"], dtype=torch.bool), layer_idx=0,
        weight_path="", router_use_softmax=m["softmax"], normalize_topk_prob=m["renorm"],
        experts_are_packed=m["bits"] == 16, quantized_experts=quantized,
        gate=_linear(w["router"]) if case["call"] == "block" else None, **shared)
    if case["call"] == "block":
        return FusedMoEBlock(_RMSNorm(w["norm"]), moe)
    return moe


def _step(state):
    return [layer(*args) for layer, args in zip(state["layers"], state["args"])]


def prepare(case, seed):
    m = MODELS[case["model"]]
    state = {"layers": [], "args": []}
    for i in range(case["layers"]):
        g = _seeded(case, seed, i)
        w = _weights(m, g)
        x, logits = _inputs(case, m, w, g)
        state["layers"].append(_module(case, m, w))
        state["args"].append((x,) if case["call"] == "block" else (x, logits))
        # the program's warm-up call: ingests the weights and sizes the workspace
        state["layers"][-1](*(torch.zeros_like(a) for a in state["args"][-1]))
    if case["replay"]:
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["out"] = _step(state)
    return state


@torch.no_grad()
def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _step(state)


# ------------------------------------------------------------------ what a pass cannot do without
def _active_experts(m, tokens, zipf):
    """Mean number of distinct experts that `tokens` tokens choose."""
    r = np.random.RandomState(7)
    spread = STD * math.sqrt(m["H"])
    bias = zipf * np.log(np.arange(m["E"]) + 1.0)
    seen = [np.unique(np.argsort(bias - spread * r.standard_normal((tokens, m["E"])), axis=1)[:, :m["k"]]).size
            for _ in range(8 if tokens <= 256 else 1)]
    return float(np.mean(seen))


def work(case):
    m, T = MODELS[case["model"]], case["tokens"]

    def weight_bytes(n, k):
        scales = {4: n * (k // 128) * 2, 8: n * 2, 16: 0}[m["bits"]]
        return n * k * m["bits"] // 8 + scales

    per_expert = weight_bytes(2 * m["I"], m["H"]) + weight_bytes(m["H"], m["I"])
    nbytes = _active_experts(m, T, case["zipf"]) * per_expert + 2 * T * m["H"] * 2
    nbytes += m["E"] * m["H"] * 2 + m["H"] * 2 if case["call"] == "block" else T * m["E"] * 2
    flops = 2 * T * m["k"] * 3 * m["H"] * m["I"]
    if m["Is"]:
        nbytes += weight_bytes(2 * m["Is"], m["H"]) + weight_bytes(m["H"], m["Is"]) + m["H"] * 2
        flops += 2 * T * (3 * m["H"] * m["Is"] + m["H"])
    if case["call"] == "block":
        flops += 2 * T * m["H"] * m["E"]
    return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * flops}


def tolerance(case):
    """bf16 hidden states and outputs: about four times the relative error against ``exact``."""
    return {"rel": 1e-2, "max": 0.1}


# ------------------------------------------------------------------ the same in 64 bits
def _swiglu(x, gate_up, down, width):
    y = x @ gate_up.T
    g, u = y[:, :width], y[:, width:]
    return (g * torch.sigmoid(g) * u) @ down.T


def _exact_layer(case, m, w, x, logits):
    """The layer on float64 values.  What the model defines in the hidden states' dtype is rounded to
    it: the normalised input, the router's logits, its probabilities and weights; of equal ones the
    lower expert is chosen."""
    x64 = x.double()
    residual = None
    if case["call"] == "block":
        residual = x64
        n = (x64 * torch.rsqrt(x64.pow(2).mean(dim=1, keepdim=True) + EPS)).to(torch.bfloat16)
        x64 = (n.double() * w["norm"].double()).to(torch.bfloat16).double()
        logits = (x64 @ w["router"].double().T).to(torch.bfloat16)
    l64 = logits.double()
    score = torch.softmax(l64, dim=1).to(torch.bfloat16).double() if m["softmax"] else l64
    ids = torch.sort(score, dim=1, descending=True, stable=True).indices[:, :m["k"]]
    p = score.gather(1, ids)
    if not m["softmax"]:
        p = torch.softmax(p, dim=1).to(torch.bfloat16).double()
    elif m["renorm"]:
        p = (p / p.sum(dim=1, keepdim=True).to(torch.bfloat16).double()).to(torch.bfloat16).double()
    out = torch.zeros_like(x64)
    for e in range(m["E"]):
        t, slot = torch.nonzero(ids == e, as_tuple=True)
        if t.numel():
            y = _swiglu(x64[t], _dense(w["gate_up"], e), _dense(w["down"], e), m["I"])
            out.index_add_(0, t, y * p[t, slot].unsqueeze(1))
    if m["Is"]:
        y = _swiglu(x64, _dense(w["shared_gate_up"], 0), _dense(w["shared_down"], 0), m["Is"])
        out += torch.sigmoid(x64 @ w["shared_gate"].double().T) * y
    return out if residual is None else out + residual


@torch.no_grad()
def exact(case, seed):
    m = MODELS[case["model"]]
    out = []
    for i in range(case["layers"]):
        g = _seeded(case, seed, i)
        w = _weights(m, g)
        x, logits = _inputs(case, m, w, g)
        out.append(_exact_layer(case, m, w, x, logits))
    return out
