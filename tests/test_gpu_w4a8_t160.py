"""160-token blocks of int4 weights with K-group scales (the tile table's pick around 128 slots per expert), whole path, bit for bit
against the CPU oracle: every fill level of a block, one and several K blocks, the three scale orders' dispatch, an expert-parallel
share, and scales that the fold without a conversion does not take."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def run(oracle, H, I, ids, E, Eg=None, flags=0, factor=1.0, scale=1.0, dtype=torch.bfloat16, named=True, **kw):
    from lightop_amd import _lib, workloads as wl
    from lightop_amd.moe import fused_experts_impl_w4a8, preshuffle_moe_scale_int4, preshuffle_moe_weight_int4

    dev = torch.device("cuda:0")
    M, k = ids.shape
    layer = wl.MoeLayer("w4-160", E=E, E_global=Eg or E, top_k=k, H=H, I=I, routing="softmax", weight_bits=4)
    t1, t2 = _lib.LoMoeTile(), _lib.LoMoeTile()
    assert _lib.lib().lo_moe_tile_query_path(_lib.LO_FORM_W4, flags, _lib.LO_BF16, 0, M, E, layer.E_global, k, H, I, t1, t2) == 0
    if named:
        assert t1.block_size_m == 160 == t2.block_size_m and t1.kernel == _lib.LO_KERNEL_T128 == t2.kernel
    w1, w2, w1s, w2s = wl.make_weights(layer, seed=M)
    x, tw, _ = wl.make_inputs(layer, M, seed=M)
    x[::7] *= scale
    x = x.to(dtype)
    w1s = w1s / scale
    emap = wl.expert_map_for(layer)
    cache13 = torch.empty(M * k * max(2 * I, H), dtype=dtype, device=dev)
    out = fused_experts_impl_w4a8(x.to(dev), preshuffle_moe_weight_int4(w1.to(dev)), preshuffle_moe_weight_int4(w2.to(dev)),
                                  tw.to(dev), ids.to(dev), cache13, global_num_experts=layer.E_global,
                                  expert_map=None if emap is None else emap.to(dev),
                                  w1_scale=preshuffle_moe_scale_int4(w1s.to(dev)), w2_scale=preshuffle_moe_scale_int4(w2s.to(dev)),
                                  block_shape=[1, 128], routed_scaling_factor=factor, lightop_amd_flags=flags, **kw)
    torch.cuda.synchronize()
    with oracle.scale_order("separate" if flags & _lib.LO_GEMM_SEPARATE_ORDER else "contract"):
        ref = oracle.fused_experts_w4a8(x, w1, w2, w1s, w2s, tw, ids, 16, global_num_experts=layer.E_global, expert_map=emap,
                                        routed_scaling_factor=factor)
    return out.cpu(), ref


@pytest.mark.parametrize("count", [1, 32, 33, 64, 65, 96, 97, 127, 128, 129, 144, 145, 159, 160, 161, 225])
@pytest.mark.parametrize("H,I", [(128, 128), (384, 256)])
def test_fill_levels(oracle, count, H, I):
    print(f"[case] int4 160-token blocks, {count} tokens on expert 0, H={H} I={I}", flush=True)
    ids = torch.ones(240, 1, dtype=torch.int32)
    ids[torch.randperm(240, generator=torch.Generator().manual_seed(count))[:count]] = 0
    out, ref = run(oracle, H, I, ids, 2)
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("what", ["separate", "fused scale", "share", "large rows", "wide"])
def test_forms(oracle, what):
    from lightop_amd import _lib

    print(f"[case] int4 160-token blocks, {what}", flush=True)
    g = torch.Generator().manual_seed(5)
    if what == "share":  # a quarter of the experts, two slots a token
        ids = torch.stack([torch.randperm(8, generator=g)[:2] for _ in range(480)]).to(torch.int32)
        out, ref = run(oracle, 512, 384, ids, 2, Eg=8, factor=2.5)
    else:
        ids = torch.randint(0, 2, (240, 1), generator=g, dtype=torch.int32)
        H, I = (1088 // 64 * 128, 640) if what == "wide" else (512, 384)
        flags = {"separate": _lib.LO_GEMM_SEPARATE_ORDER, "fused scale": _lib.LO_GEMM_FUSED_SCALE}.get(what, 0)
        out, ref = run(oracle, H, I, ids, 2, flags=flags, scale=2.0 ** 56 if what == "large rows" else 1.0)
    assert bool(ref.float().isfinite().all())
    if what == "fused scale":  # against the default order: last-ulp differences in fp32, which move some values of the second quantisation
        err, ref = (out.float() - ref.float()).abs(), ref.float().abs()  # by a step of 1 / 127 of their group's largest: bounds of the path
        assert err.max() <= 1e-2 * ref.max() and err.sum() <= 2e-3 * ref.sum()
        return
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("tokens", [9, 240, 700])
def test_as_the_caller_asks(oracle, tokens):
    """Taken where the table names it, refused beside."""
    print(f"[case] int4 160-token blocks on request, {tokens} tokens", flush=True)
    ids = torch.randint(0, 2, (tokens, 1), generator=torch.Generator().manual_seed(tokens), dtype=torch.int32)
    if tokens != 240:
        with pytest.raises(RuntimeError, match="block_size_m 160"):
            run(oracle, 384, 256, ids, 2, named=False, lightop_amd_block_size_m=160)
        return
    out, ref = run(oracle, 384, 256, ids, 2, lightop_amd_block_size_m=160)
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))


def test_in_chunks(oracle, monkeypatch):
    """A call that the table names 160 for, cut into chunks that it names other sizes for."""
    print("[case] int4 160-token blocks on request, two chunks", flush=True)
    ids = torch.randint(0, 2, (240, 1), generator=torch.Generator().manual_seed(6), dtype=torch.int32)
    monkeypatch.setenv("LMSLIM_FUSED_MOE_CHUNK_SIZE", "200")
    out, ref = run(oracle, 384, 256, ids, 2, lightop_amd_block_size_m=160)
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("tokens", [100, 240])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_from_a_tuning_file(oracle, monkeypatch, tmp_path, dtype, tokens):
    """A file's 160 is taken by a call that can, and left to the table by one that cannot."""
    import json

    from lightop_amd.moe import tile_files

    print(f"[case] int4 160-token blocks from a file, {dtype}, {tokens} tokens", flush=True)
    cfg = {"BLOCK_SIZE_M": 160}
    with open(tmp_path / tile_files.file_name(2, 512, 384, 256, 1, [1, 128], True), "w") as f:
        json.dump({"512_384_256": {"64": {"config1": cfg, "config2": cfg}}}, f)
    monkeypatch.setenv("TRITON_JSON_DIR", str(tmp_path))
    tile_files.forget()
    ids = torch.randint(0, 2, (tokens, 1), generator=torch.Generator().manual_seed(3), dtype=torch.int32)
    assert tile_files.block_size_m(tokens, 2, 512, 384, 256, 1, [1, 128], int4=True) == 160
    out, ref = run(oracle, 384, 256, ids, 2, dtype=dtype, named=False)
    tile_files.forget()
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))


def test_stages(oracle):
    """The stage entry points take the size the tile table names."""
    from lightop_amd import _lib, workloads as wl
    from lightop_amd.moe import (invoke_fused_moe_gemm1_silu_quant, invoke_fused_moe_kernel_int8, moe_align_block_size,
                                 preshuffle_moe_scale_int4, preshuffle_moe_weight_int4)
    from lightop_amd.quant import per_token_group_quant_int8

    dev = torch.device("cuda:0")
    layer = wl.MoeLayer("w4-160", E=3, E_global=3, top_k=2, H=512, I=256, routing="softmax", weight_bits=4)
    weights, inputs = wl.make_weights(layer, seed=1), wl.make_inputs(layer, 300, seed=1)
    w1, w2, w1s, w2s = weights
    x, tw, ids = inputs
    rs, re, rp = oracle.moe_align_block_size(ids, 16, 3)
    aq, asc = oracle.per_token_group_quant_int8(x)
    rq, rsc = oracle.per_token_group_quant_int8(oracle.silu_and_mul(oracle.moe_gemm_w4a8(aq, asc, w1, w1s, rs, re, rp, tw, False, 2, 600, 16)))
    rC = oracle.moe_gemm_w4a8(rq, rsc, w2, w2s, rs, re, rp, tw, True, 1, 600, 16)
    w1, w2, w1s, w2s = (t.to(dev) for t in weights)
    x, tw, ids = (t.to(dev) for t in inputs)
    xq, xs = per_token_group_quant_int8(x, 128)
    for bs in (160, 128):
        print(f"[case] int4 stages, block {bs}", flush=True)
        s, e, p = moe_align_block_size(ids, bs, 3)
        q, sc = invoke_fused_moe_gemm1_silu_quant(xq, preshuffle_moe_weight_int4(w1), xs, preshuffle_moe_scale_int4(w1s), tw, s, e, p,
                                                  False, 2, 600, {"BLOCK_SIZE_M": bs}, flags=_lib.LO_GEMM_W4)
        C = torch.empty(300, 2, 512, dtype=torch.bfloat16, device=dev)
        invoke_fused_moe_kernel_int8(q, preshuffle_moe_weight_int4(w2), C, sc, preshuffle_moe_scale_int4(w2s), tw, s, e, p, True, 1,
                                     {"BLOCK_SIZE_M": bs}, flags=_lib.LO_GEMM_W4)
        torch.cuda.synchronize()
        assert torch.equal(q.cpu(), rq) and torch.equal(sc.cpu(), rsc)
        assert torch.equal(C.view(600, 512).cpu().view(torch.int16), rC.view(torch.int16))
