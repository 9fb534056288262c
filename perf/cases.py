"""The work this package is used for, as cases to measure.

A case is one pass of a routed MoE layer as a serving program runs it: the router on the gate's logits
(``topk_softmax`` or ``moe_fused_gate``), then the experts (``fused_experts_impl_int8`` or
``fused_experts_impl_w4a8``) on the routing it wrote.  The layers are the ones of
``lightop_amd.workloads``; token counts run from one (a single sequence decoding) over decode batches
and chunked prefill to 8192 tokens.  What a program holds before the call - weights in their load-time
layout, the process-wide workspace, the step's activations and logits - is made by ``prepare``.

``activation``, ``dtype`` and ``rows`` (weights kept row-major, as a checkpoint holds them, by a program
that only swapped the import) are the options such programs choose among.
"""
from __future__ import annotations

import dataclasses
import functools
import math

import torch

from lightop_amd import workloads as wl
from lightop_amd.moe import (fused_experts_impl_int8, fused_experts_impl_w4a8, get_moe_cache, moe_fused_gate,
                             preshuffle_moe_scale_int4, preshuffle_moe_weight, preshuffle_moe_weight_int4, topk_softmax)

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}

MAX_TOKENS = 8192


def _case(name, layer, tokens, dtype="bf16", activation="silu", rows=False):
    c = {"layer": layer, "tokens": tokens, "dtype": dtype, "activation": activation, "rows": rows}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one sequence decoding: the latency of the launches and of the host path around them
        _case("block, decode 1", "qwen3-30b-a3b", 1),
        # a decode batch of a server
        _case("block, decode 24", "qwen3-30b-a3b", 24),
        # a chunk of prefill with decode tokens riding along
        _case("block, chunk 1531", "qwen3-30b-a3b", 1531),
        # the largest prefill batch
        _case("block, prefill 8192", "qwen3-30b-a3b", 8192),
        # an expert-parallel rank: 32 of 256 experts, grouped gate, shared expert added in the reduction
        _case("block, rank of 8, decode 64", "deepseek-v3-ep8-share", 64),
        _case("block, rank of 8, prefill 4096", "deepseek-v3-ep8-share", 4096),
        # every expert on one GPU, skewed routing
        _case("block, all experts, 8192", "deepseek-v3-full", 8192),
        # weights as the checkpoint holds them
        _case("block, row-major, 200", "qwen3-235b-a22b", 200, rows=True),
        # int4 weights with K-group scales
        _case("int4 groups, 2048", "qwen3-235b-a22b-w4a8", 2048),
        # int4 weights with one scale per row
        _case("int4 channels, decode 37", "qwen3-235b-a22b-w4a8-channel", 37),
        # int8 weights with one scale per row
        _case("int8 channels, 700", "qwen3-30b-a3b-channel", 700),
        # a model served in half precision
        _case("block, fp16, 333", "qwen3-30b-a3b", 333, dtype="fp16"),
    ]


# layer and how often it is drawn
_DRAWN = (("qwen3-30b-a3b", 4), ("deepseek-v3-ep8-share", 3), ("deepseek-v3-full", 1), ("qwen3-235b-a22b", 2),
          ("qwen3-235b-a22b-w4a8", 2), ("qwen3-235b-a22b-w4a8-channel", 2), ("qwen3-30b-a3b-channel", 2),
          ("deepseek-v3-ep8-share-channel", 1))


def draw(rng):
    layer = rng.choices([n for n, _ in _DRAWN], [w for _, w in _DRAWN])[0]
    tokens = min(MAX_TOKENS, max(1, round(math.exp(rng.uniform(0.0, math.log(MAX_TOKENS + 1))))))
    dtype = "fp16" if rng.random() < 0.15 else "bf16"
    activation = "gelu" if rng.random() < 0.08 else "silu"
    rows = wl.LAYERS[layer].weight_bits == 8 and rng.random() < 0.12
    return _case(None, layer, tokens, dtype, activation, rows)


def prepare(case, seed):
    layer, M = wl.LAYERS[case["layer"]], int(case["tokens"])
    dev, dtype = torch.device("cuda:0"), DTYPES[case["dtype"]]
    w1, w2, w1s, w2s = wl.make_weights(layer, seed=seed, device=dev, gen_device="cuda")
    if layer.weight_bits == 4:
        w1, w2 = preshuffle_moe_weight_int4(w1), preshuffle_moe_weight_int4(w2)
        if layer.quant != "channel":
            w1s, w2s = preshuffle_moe_scale_int4(w1s), preshuffle_moe_scale_int4(w2s)
    elif not case["rows"]:
        w1, w2 = preshuffle_moe_weight(w1), preshuffle_moe_weight(w2)

    g = torch.Generator(device=dev).manual_seed(seed * 7919 + M)

    def normal(*shape):
        return torch.randn(shape, generator=g, dtype=torch.float32, device=dev)

    logits = normal(M, layer.E_global)
    s = {"layer": layer, "x": normal(M, layer.H).to(dtype), "w1": w1, "w2": w2, "w1s": w1s, "w2s": w2s,
         "emap": wl.expert_map_for(layer, dev), "activation": case["activation"],
         "cache13": get_moe_cache(layer.top_k, 2 * layer.I, layer.H, dev, dtype)}
    if layer.routing == "softmax":
        s["logits"] = logits.to(dtype)  # the gate is a linear layer of the model's own type
        return s
    if layer.routing.endswith("zipf"):  # exponent 1.2 over a random order of the experts
        rank = torch.arange(1, layer.E_global + 1, dtype=torch.float32, device=dev)
        logits[:, torch.randperm(layer.E_global, generator=g, device=dev)] -= 1.2 * torch.log(rank)
    s["logits"] = logits  # grouped gates are kept in fp32
    s["bias"] = 0.01 * normal(layer.E_global)
    s["shared"] = normal(M, layer.H).to(dtype)
    return s


def run(s):
    layer, x, logits = s["layer"], s["x"], s["logits"]
    factor, shared = 1.0, None
    if layer.routing == "softmax":
        weights = torch.empty(x.shape[0], layer.top_k, dtype=torch.float32, device=x.device)
        ids = torch.empty(x.shape[0], layer.top_k, dtype=torch.int32, device=x.device)
        topk_softmax(weights, ids, None, logits, True)
    else:
        factor, shared = layer.routed_scaling, s["shared"]
        weights, ids = moe_fused_gate(logits, s["bias"], layer.n_group, layer.topk_group, layer.top_k, 0, factor,
                                      apply_routed_scaling_factor_on_output=False)
    if layer.weight_bits == 4:
        out = fused_experts_impl_w4a8(
            x, s["w1"], s["w2"], weights, ids, s["cache13"], activation=s["activation"],
            global_num_experts=layer.E_global, expert_map=s["emap"], w1_scale=s["w1s"], w2_scale=s["w2s"],
            block_shape=None if layer.quant == "channel" else [1, 128], routed_scaling_factor=factor,
            shared_output=shared)
    else:
        channel = layer.quant == "channel"
        out = fused_experts_impl_int8(
            x, s["w1"], s["w2"], weights, ids, s["cache13"], activation=s["activation"], use_int8_w8a8=True,
            per_channel_quant=channel, global_num_experts=layer.E_global, expert_map=s["emap"], w1_scale=s["w1s"],
            w2_scale=s["w2s"], block_shape=None if channel else [128, 128], routed_scaling_factor=factor,
            shared_output=shared)
    return {"out": out, "weights": weights, "ids": ids}


@functools.lru_cache(maxsize=None)
def _zipf_shares(name):
    """Share of the tokens that every expert of a layer with skewed routing sees (a fixed sample of tokens)."""
    layer = wl.LAYERS[name]
    _, _, ids = wl.make_inputs(dataclasses.replace(layer, H=128), 4096, seed=1)
    return torch.bincount(ids.reshape(-1).long(), minlength=layer.E_global).double() / ids.shape[0]


def _experts_hit(layer, M):
    """Experts with at least one slot, on average."""
    if layer.routing.endswith("zipf"):
        return float((1.0 - (1.0 - _zipf_shares(layer.name)) ** M).sum())
    return layer.E * (1.0 - (1.0 - layer.top_k / layer.E_global) ** M)


def work(case):
    """Weights and scales of the experts that are hit, logits, activations in and out; the products of every
    routed slot of a resident expert."""
    layer, M = wl.LAYERS[case["layer"]], int(case["tokens"])
    E, Eg, k, H, I = layer.E, layer.E_global, layer.top_k, layer.H, layer.I
    hit = _experts_hit(layer, M)
    weights = 3 * I * H * layer.weight_bits // 8
    if layer.quant == "channel":
        scales = 4 * (2 * I + H)
    elif layer.weight_bits == 4:
        scales = 4 * (2 * I * (H // 128) + H * (I // 128))
    else:
        scales = 4 * ((2 * I // 128) * (H // 128) + (H // 128) * (I // 128))
    softmax = layer.routing == "softmax"
    rows = 2 if softmax else 3  # hidden states in, out, and the shared expert's output
    nbytes = hit * (weights + scales) + rows * 2 * M * H + M * Eg * (2 if softmax else 4) + 8 * M * k
    return {"bytes": float(nbytes), "flops": 6.0 * M * k * E / Eg * I * H}


def tolerance(case):
    # 16-bit results of 32-bit sums, with two roundings to int8 on the way whose inputs the order of those sums
    # can move across a step; router weights and ids are 32-bit arithmetic with ties going to the lower id
    return {"rel": 5e-3, "max": 0.1}
