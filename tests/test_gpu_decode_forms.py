"""The two-launch path for every form, row type and activation, bit for bit against the staged path: one to seven K blocks
per wave, ranks that hold a part of the experts, experts with more slots than one pass multiplies, more experts hit than
the grid has rows, shared-expert epilogue and router weight on the input."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def make_layer(form, activation, name, E, Eg, k, H, I):
    """The layer, and its entry point with the weights and scales bound."""
    from lightop_amd import workloads as wl
    from lightop_amd.moe import (fused_experts_impl_int8, fused_experts_impl_w4a8, preshuffle_moe_scale_int4,
                                 preshuffle_moe_weight, preshuffle_moe_weight_int4)

    dev = torch.device("cuda:0")
    extra = {"quant": "channel"} if form.endswith("channel") else {}
    if form.startswith("w4"):
        extra["weight_bits"] = 4
    layer = wl.MoeLayer(name, E=E, E_global=Eg, top_k=k, H=H, I=I, routing="softmax", **extra)
    w1, w2, w1s, w2s = wl.make_weights(layer, seed=3, device=dev)
    kw = dict(w1_scale=w1s, w2_scale=w2s, activation=activation, global_num_experts=Eg,
              block_shape=None if "channel" in form else [1, 128] if form == "w4" else [128, 128])
    if form.startswith("w4"):
        fn, w1, w2 = fused_experts_impl_w4a8, preshuffle_moe_weight_int4(w1), preshuffle_moe_weight_int4(w2)
        if form == "w4":
            kw.update(w1_scale=preshuffle_moe_scale_int4(w1s), w2_scale=preshuffle_moe_scale_int4(w2s))
    else:
        fn, w1, w2 = fused_experts_impl_int8, preshuffle_moe_weight(w1), preshuffle_moe_weight(w2)
        kw.update(use_int8_w8a8=True, per_channel_quant=form == "channel")

    def run(x, tw, ids, cache13, **kx):
        return fn(x, w1, w2, tw, ids, cache13, **kw, **kx)

    return layer, run


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("activation", ["silu", "gelu"])
@pytest.mark.parametrize("form", ["block", "channel", "w4", "w4_channel"])
@pytest.mark.parametrize("shape", ["one", "share", "seven", "wide", "crowded"])
def test_forms(form, activation, dtype, shape):
    from lightop_amd import _lib, workloads as wl

    E, Eg, k, H, I, tokens = {"one": (8, 8, 2, 128, 128, (1, 3)), "share": (4, 32, 8, 1024, 896, (1, 5, 9)),
                              "seven": (4, 4, 2, 3584, 256, (1, 2, 16)), "wide": (3, 3, 1, 2560, 2304, (1, 4)),
                              "crowded": (3, 6, 3, 256, 128, (21, 50))}[shape]
    dev = torch.device("cuda:0")
    layer, run = make_layer(form, activation, shape, E, Eg, k, H, I)
    for M in tokens:
        print(f"[case] decode forms {form} {activation} {dtype} {shape} M={M}", flush=True)
        x, tw, ids = (t.to(dev) for t in wl.make_inputs(layer, M, seed=M))
        x = x.to(dtype)
        x[M // 2] = 0
        emap = None
        if E != Eg:
            emap = torch.full((Eg,), -1, dtype=torch.int32, device=dev)
            emap[torch.randperm(Eg, generator=torch.Generator().manual_seed(1))[:E].to(dev)] = torch.arange(
                E, dtype=torch.int32, device=dev)
        outs = []
        for flag in (_lib.LO_FUSED_NO_DECODE_PATH, _lib.LO_FUSED_FORCE_DECODE_PATH):
            cache13 = torch.full((M * k * max(2 * I, H),), float("nan"), dtype=dtype, device=dev)
            kx = dict(shared_output=x + 1, routed_scaling_factor=2.5) if M % 2 else {}
            outs.append(run(x, tw, ids, cache13, expert_map=emap, lightop_amd_flags=flag,
                            apply_router_weight_on_input=M == tokens[-1], **kx).cpu())
            if flag == _lib.LO_FUSED_FORCE_DECODE_PATH:  # only this path leaves the activations at the front of the cache
                act = cache13[: M * k * I].view(M * k, I).cpu()
                here = ids.reshape(-1) if emap is None else emap[ids.reshape(-1).long()]
                assert not torch.isnan(act[(here >= 0).cpu()].float()).any()
        assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16)), f"M={M}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H", [256, 3584])  # one K block per wave, several
@pytest.mark.parametrize("form", ["block", "channel", "w4", "w4_channel"])
@pytest.mark.parametrize("routing", ["twice", "all equal", "many to one", "few finite logits"])
def test_one_token_with_a_repeated_expert(form, H, dtype, routing):
    """One token, several of its slots on one local expert: a caller's own ids, more of them than a pass multiplies, a map
    that sends several global ids to one expert, and the router on a row with fewer finite logits than picks.  A first
    pass with large rows leaves its values in the registers that a row which is not loaded would be read from."""
    from lightop_amd import _lib, workloads as wl
    from lightop_amd.moe import topk_softmax

    dev, k = torch.device("cuda:0"), 2 if routing == "twice" else 6
    E, Eg = (4, 8) if routing == "many to one" else (8, 8)
    print(f"[case] one token, repeated expert {form} H={H} {dtype} {routing}", flush=True)
    layer, run = make_layer(form, "silu", "repeated", E, Eg, k, H, 256)
    x, tw, ids = (t.to(dev) for t in wl.make_inputs(layer, 1, seed=11))
    x, emap = x.to(dtype), None
    if routing == "twice":
        ids.fill_(3)
    elif routing == "all equal":
        ids.fill_(5)
    elif routing == "many to one":
        emap = torch.tensor([2, 2, -1, 0, 2, 0, 2, 1], dtype=torch.int32, device=dev)
        ids.copy_(torch.tensor([[0, 4, 1, 2, 6, 3]], device=dev))
    else:
        logits = torch.full((1, Eg), float("-inf"), device=dev)
        logits[0, 6] = logits[0, 2] = 1.0
        topk_softmax(tw, ids, None, logits, True)
        assert ids.flatten().bincount(minlength=Eg).max() > 1
    outs = []
    for flag in (_lib.LO_FUSED_NO_DECODE_PATH, _lib.LO_FUSED_FORCE_DECODE_PATH):
        cache13 = torch.full((k * max(2 * 256, H),), float("nan"), dtype=dtype, device=dev)
        other = torch.full((8, H), 1e4, dtype=dtype, device=dev)
        run(other, tw.expand(8, k).contiguous(), ids.expand(8, k).contiguous(), torch.empty(8 * cache13.numel(), dtype=dtype, device=dev),
            expert_map=emap, lightop_amd_flags=flag)
        outs.append(run(x, tw, ids, cache13, expert_map=emap, lightop_amd_flags=flag).cpu())
    assert torch.isfinite(outs[0].float()).all()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("activation", ["silu", "gelu"])
@pytest.mark.parametrize("form", ["block", "channel", "w4", "w4_channel"])
def test_tile_query_names_the_path_that_is_taken(form, activation, dtype):
    """On both sides of every form's line between the two-launch path, which leaves the workspace alone, and the
    staged path, which does not."""
    from lightop_amd import workloads as wl
    from lightop_amd.moe import get_w8a8moe_json

    dev, k, (E, H, I) = torch.device("cuda:0"), 8, (16, 1024, 256)
    layer, run = make_layer(form, activation, "query", E, E, k, H, I)
    block_shape = None if "channel" in form else [1, 128] if form == "w4" else [128, 128]
    taken = []
    for M in (1, 2, 3, 4, 5, 8, 9):
        print(f"[case] tile query {form} {activation} {dtype} M={M}", flush=True)
        x, tw, ids = (t.to(dev) for t in wl.make_inputs(layer, M, seed=M))
        cache13 = torch.empty(M * k * max(2 * I, H), dtype=dtype, device=dev)
        ws = torch.full((1 << 20,), 0xA5, dtype=torch.uint8, device=dev)
        run(x.to(dtype), tw, ids, cache13, lightop_amd_workspace=ws)
        kernel = get_w8a8moe_json(M, E, 2 * I, H, I, True, block_shape, k, E, int4=form.startswith("w4"), dtype=dtype,
                                  activation=activation)[0]["kernel_name"]
        taken.append(bool((ws == 0xA5).all()))
        assert taken[-1] == kernel.startswith("dec_"), (M, kernel)
    assert taken[0] and not taken[-1]
