"""The looked-up activations of the fused first stage (GELU; SiLU of fp16 rows) at the edges of its dispatch, bit for bit
against the launches they replace (which another scale order or forced streaming still takes): block sizes, both weight
layouts and packed int4, blocks with one token, one short of full and one over, gates that overflow or are NaN."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,activation", [(torch.float16, "silu"), (torch.float16, "gelu"), (torch.bfloat16, "gelu")])
@pytest.mark.parametrize("form", ["rows", "block", "w4"])
@pytest.mark.parametrize("bs", [16, 32, 64, 128])
def test_fused_act(form, bs, dtype, activation):
    from lightop_amd import _lib, workloads as wl
    from lightop_amd.moe import (fused_experts_impl_int8, fused_experts_impl_w4a8,
                                 fused_experts_workspace_bytes, fused_experts_workspace_views,
                                 preshuffle_moe_scale_int4, preshuffle_moe_weight, preshuffle_moe_weight_int4)

    dev = torch.device("cuda:0")
    layer = wl.MoeLayer("edge", E=4, E_global=4, top_k=1, H=384, I=256, routing="softmax",
                        **({"weight_bits": 4} if form == "w4" else {}))
    w1, w2, w1s, w2s = wl.make_weights(layer, seed=bs, device=dev)
    w1s[0] *= 1e6  # expert 0: gates and products that leave the 16-bit range
    counts = [1, bs - 1, bs, bs + 1]
    ids = torch.repeat_interleave(torch.arange(4, dtype=torch.int32), torch.tensor(counts)).view(-1, 1).to(dev)
    M = ids.shape[0]
    print(f"[case] fused activation {form} bs={bs} {dtype} {activation} M={M}", flush=True)
    x, tw, _ = (t.to(dev) for t in wl.make_inputs(layer, M, seed=1))
    x = x.to(dtype)
    kw = dict(w1_scale=w1s, w2_scale=w2s, activation=activation, block_shape=[1, 128] if form == "w4" else [128, 128])
    fn = fused_experts_impl_int8
    if form == "w4":
        fn, w1, w2 = fused_experts_impl_w4a8, preshuffle_moe_weight_int4(w1), preshuffle_moe_weight_int4(w2)
        kw.update(w1_scale=preshuffle_moe_scale_int4(w1s), w2_scale=preshuffle_moe_scale_int4(w2s))
    else:
        kw.update(use_int8_w8a8=True)
        if form == "block":
            w1, w2 = preshuffle_moe_weight(w1), preshuffle_moe_weight(w2)
    got = []
    for flag in (0, _lib.LO_GEMM_FORCE_STREAMING):
        ws = torch.zeros(fused_experts_workspace_bytes(M, 1, layer.H, layer.I, 4) + 256, dtype=torch.uint8, device=dev)
        cache13 = torch.empty(M * max(2 * layer.I, layer.H), dtype=dtype, device=dev)
        fn(x, w1, w2, tw, ids, cache13, lightop_amd_workspace=ws, lightop_amd_block_size_m=bs, lightop_amd_flags=flag,
           apply_router_weight_on_input=bs == 32, **kw)
        torch.cuda.synchronize()
        v = fused_experts_workspace_views(ws, M, 1, layer.H, layer.I, 4, bs)
        got.append((v["a2q"].clone(), v["a2s"].clone()))
    assert torch.equal(got[0][0], got[1][0])
    assert torch.equal(got[0][1].view(torch.int32), got[1][1].view(torch.int32))


@pytest.mark.parametrize("dtype,activation", [(torch.bfloat16, "silu"), (torch.float16, "silu"), (torch.bfloat16, "gelu")])
@pytest.mark.parametrize("form", ["rows", "int8", "w4"])
@pytest.mark.parametrize("bs", [64, 128, 160])
def test_gated_channel(form, bs, dtype, activation):
    """The per-channel first stage that ends with the activation in 16 bits, against the plain one and the activation launch."""
    from lightop_amd import _lib, workloads as wl
    from lightop_amd.moe import (fused_experts_impl_int8, fused_experts_impl_w4a8, fused_experts_workspace_bytes,
                                 fused_experts_workspace_views, preshuffle_moe_weight, preshuffle_moe_weight_int4)

    if form == "rows" and bs == 160:
        pytest.skip("row-major weights have no 160-token blocks")
    dev = torch.device("cuda:0")
    layer = wl.MoeLayer("edge", E=4, E_global=5, top_k=1, H=384, I=256, routing="softmax", quant="channel",
                        **({"weight_bits": 4} if form == "w4" else {}))
    w1, w2, w1s, w2s = wl.make_weights(layer, seed=bs, device=dev)
    w1s[0] *= 1e6
    counts = [1, bs - 1, bs, bs + 1, 3]
    ids = torch.repeat_interleave(torch.arange(5, dtype=torch.int32), torch.tensor(counts)).view(-1, 1).to(dev)
    M = ids.shape[0]
    print(f"[case] gated channel {form} bs={bs} {dtype} {activation} M={M}", flush=True)
    x, tw, _ = (t.to(dev) for t in wl.make_inputs(layer, M, seed=1))
    x = x.to(dtype)
    x[M // 2] = 0
    emap = torch.tensor([0, 1, 2, 3, -1], dtype=torch.int32, device=dev)
    kw = dict(w1_scale=w1s, w2_scale=w2s, activation=activation, block_shape=None, expert_map=emap, global_num_experts=5)
    fn = fused_experts_impl_int8
    if form == "w4":
        fn, w1, w2 = fused_experts_impl_w4a8, preshuffle_moe_weight_int4(w1), preshuffle_moe_weight_int4(w2)
    else:
        kw.update(use_int8_w8a8=True, per_channel_quant=True)
        if form == "int8":
            w1, w2 = preshuffle_moe_weight(w1), preshuffle_moe_weight(w2)
    got = []
    for flag, b in ((0, bs), (_lib.LO_GEMM_FORCE_STREAMING, min(bs, 128))):
        ws = torch.zeros(fused_experts_workspace_bytes(M, 1, layer.H, layer.I, 5) + 256, dtype=torch.uint8, device=dev)
        cache13 = torch.empty(M * max(2 * layer.I, layer.H), dtype=dtype, device=dev)
        out = fn(x, w1, w2, tw, ids, cache13, lightop_amd_workspace=ws, lightop_amd_block_size_m=b, lightop_amd_flags=flag,
                 apply_router_weight_on_input=bs == 128, **kw)
        torch.cuda.synchronize()
        v = fused_experts_workspace_views(ws, M, 1, layer.H, layer.I, 5, b)
        here = M - counts[-1]
        got.append((v["a2q"][:here].clone(), v["a2s"].view(-1)[:here].view(torch.int32).clone(), out.view(torch.int16)))
    for a, b in zip(*got):
        assert torch.equal(a, b)
