"""Host-side logic that needs no GPU: the Python drop-in surface, lazy flags, workload
generators and the golden fixtures against the oracle."""
import hashlib
import importlib
import inspect
import json
import os

import numpy as np
import pytest
import torch

HERE = os.path.dirname(os.path.abspath(__file__))
GOLDEN = os.path.join(HERE, "golden")


def test_import_touches_no_gpu_and_surface_matches_the_reference():
    import lightop_amd
    from lightop_amd import moe, quant

    assert {"fused_experts_impl_int8", "moe_align_block_size", "moe_align_block_size_out", "moe_sum"} <= set(moe.__all__)
    assert "per_token_group_quant_int8" in quant.__all__
    # the quant entry point stays out of the moe namespace (reference: test_quant_per_token_quant_int8.py:22-25)
    assert "per_token_group_quant_int8" not in moe.__all__
    assert lightop_amd.moe_sum is moe.moe_sum
    with pytest.raises(AttributeError):
        moe.no_such_function


def test_signatures_match_the_reference():
    from lightop_amd import moe, quant

    sig = inspect.signature(moe.fused_experts_impl_int8)
    names = list(sig.parameters)
    # int8.py:628-656
    assert names[:6] == ["hidden_states", "w1", "w2", "topk_weights", "topk_ids", "cache13"]
    assert names[6:] == ["inplace", "activation", "apply_router_weight_on_input", "use_fp8_w8a8", "use_int8_w8a8",
                         "use_int8_w8a16", "use_int4_w4a16", "per_channel_quant", "global_num_experts", "expert_map",
                         "w1_scale", "w2_scale", "w1_zp", "w2_zp", "a1_scale", "a2_scale", "block_shape",
                         "use_nn_moe", "routed_scaling_factor", "shared_output", "i_q", "i_s", "_"]
    assert sig.parameters["inplace"].default is False and sig.parameters["activation"].default == "silu"
    assert sig.parameters["global_num_experts"].default == -1 and sig.parameters["routed_scaling_factor"].default == 1.0
    assert sig.parameters["_"].kind is inspect.Parameter.VAR_KEYWORD
    # moe_align_block_size.py:17-24
    assert list(inspect.signature(moe.moe_align_block_size).parameters) == [
        "topk_ids", "block_size", "num_experts", "expert_map", "pad_sorted_ids", "ignore_invalid_experts"]
    # moe/routing.py:23-35
    assert list(inspect.signature(moe.moe_align_block_size_out).parameters) == [
        "topk_ids", "num_experts", "block_size", "sorted_ids", "expert_ids", "num_tokens_post_pad", "expert_map",
        "expert_mask", "num_local_tokens", "is_ep", "is_fuse_fill"]
    # moe_align_sum.py:12-20
    ms = inspect.signature(moe.moe_sum)
    assert list(ms.parameters) == ["input", "output", "bias", "expert_mask", "num_local_tokens", "factor", "expect_m"]
    assert ms.parameters["factor"].default == 1.0 and ms.parameters["expect_m"].default == -1
    # int8_utils.py:125-130
    qs = inspect.signature(quant.per_token_group_quant_int8)
    assert list(qs.parameters) == ["x", "group_size", "eps", "dtype"]
    assert qs.parameters["eps"].default == 1e-10 and qs.parameters["dtype"].default is torch.int8
    # int8_utils.py:46
    assert list(inspect.signature(quant.per_token_quant_int8).parameters) == ["x"]
    # w4a8.py:480-501
    w4 = inspect.signature(moe.fused_experts_impl_w4a8)
    assert list(w4.parameters) == ["hidden_states", "w1", "w2", "topk_weights", "topk_ids", "cache13", "inplace",
                                   "activation", "apply_router_weight_on_input", "global_num_experts", "expert_map",
                                   "w1_scale", "w2_scale", "w1_zp", "w2_zp", "a1_scale", "a2_scale", "block_shape",
                                   "use_nn_moe", "routed_scaling_factor", "shared_output", "_"]
    # gemmopt.py:437-447 (a trailing private `flags` is this build's)
    from lightop_amd import fuse_silu_mul_quant, gemmopt, op
    from lightop_amd.moe import routing as gate_mod

    assert list(inspect.signature(gemmopt.moe_gemm_w8a8).parameters)[:11] == [
        "input", "b_qweight", "output", "a_scale", "b_scale", "topk_weights", "sorted_token_ids", "experts_ids",
        "num_tokens_post_pad", "top_k", "config"]
    # fuse_silu_mul_quant.py:45-51
    fs = inspect.signature(fuse_silu_mul_quant)
    assert list(fs.parameters) == ["input", "num_local_tokens_tensor", "topk", "expect_m", "output", "scales",
                                   "expert_ids"]
    assert fs.parameters["topk"].default == 1 and fs.parameters["expect_m"].default == -1
    # moe_fused_gate.py:10-20 and op.topk_softmax (export.cpp:1437)
    assert list(inspect.signature(gate_mod.moe_fused_gate).parameters) == [
        "x", "bias", "num_expert_group", "topk_group", "topk", "n_share_experts_fusion", "routed_scaling_factor",
        "apply_routed_scaling_factor_on_output", "output_indices_int64"]
    assert list(inspect.signature(op.topk_softmax).parameters) == [
        "topk_weights", "topk_indices", "token_expert_indices", "gating_output", "Is_renormalize"]


def test_out_variant_forwards_positionally(monkeypatch):
    """moe_align_block_size_out passes its 11 arguments through unchanged
    (reference: test/test_moe_align_block_size_out.py:11-27)."""
    from lightop_amd.moe import routing

    seen = {}
    monkeypatch.setattr(routing.op, "moe_align_block_size", lambda *a: seen.setdefault("args", a))
    routing.moe_align_block_size_out(1, 2, 3, 4, 5, 6, 7, 8, 9, True, False)
    assert seen["args"] == (1, 2, 3, 4, 5, 6, 7, 8, 9, True, False)


def test_env_flags_are_lazy(monkeypatch):
    from lightop_amd import envs

    assert envs.LMSLIM_FUSED_MOE_CHUNK_SIZE == 16 * 1024
    monkeypatch.setenv("VLLM_FUSED_MOE_CHUNK_SIZE", "4096")
    assert envs.LMSLIM_FUSED_MOE_CHUNK_SIZE == 4096
    monkeypatch.setenv("LMSLIM_FUSED_MOE_CHUNK_SIZE", "512")  # the LMSLIM name wins over the alias
    assert envs.LMSLIM_FUSED_MOE_CHUNK_SIZE == 512
    assert envs.LMSLIM_USE_GLOBAL_MOE_CACHE is False
    monkeypatch.setenv("LMSLIM_USE_GLOBAL_MOE_CACHE", "yes")
    assert envs.LMSLIM_USE_GLOBAL_MOE_CACHE is True
    with pytest.raises(AttributeError):
        envs.NOT_A_FLAG


def test_cpu_tensors_are_rejected_loudly():
    """There is no CPU fallback: a CPU tensor is an error, not a slow path."""
    from lightop_amd import moe, quant

    with pytest.raises(RuntimeError, match="GPU"):
        quant.per_token_group_quant_int8(torch.zeros(2, 128, dtype=torch.bfloat16), 128)
    with pytest.raises(RuntimeError, match="GPU"):
        moe.moe_sum(torch.zeros(2, 2, 128, dtype=torch.bfloat16), torch.zeros(2, 128, dtype=torch.bfloat16))


def test_missing_library_is_an_error(monkeypatch, tmp_path):
    from lightop_amd import _lib

    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "nope.so"))
    with pytest.raises(RuntimeError, match="no CPU or PyTorch fallback"):
        _lib.lib()


def test_product_never_imports_the_oracle():
    """The oracle is the checker; the shipped package must not reach it in any way."""
    root = os.path.dirname(HERE)
    for d, _, files in os.walk(os.path.join(root, "lightop_amd")):
        for f in files:
            if f.endswith((".py", ".hip", ".h")):
                text = open(os.path.join(d, f)).read()
                for needle in ("import oracle", "from oracle", "oracle/", "moe_oracle", "cpu_oracle", "torch_ref"):
                    assert needle not in text, f"{f} refers to {needle}"


def test_tile_config_dictionary():
    from lightop_amd.moe import get_w8a8moe_json

    c1, c2 = get_w8a8moe_json(64, 32, 4096, 7168, 2048, True, [128, 128], 8, 256)
    for c in (c1, c2):
        assert {"BLOCK_SIZE_M", "BLOCK_SIZE_N", "BLOCK_SIZE_K", "GROUP_SIZE_M", "num_warps", "num_stages"} <= set(c)
    assert c1["BLOCK_SIZE_M"] == c2["BLOCK_SIZE_M"] == 16  # the alignment block serves both GEMMs (int8.py:767)


def test_per_channel_config_lookup_mirrors_the_reference_call():
    """get_moe_cuda_config as the per-channel branch calls it (int8.py:739): two dictionaries and a status."""
    from lightop_amd.moe import get_moe_cuda_config

    E, M, H, I, k = 128, 512, 2048, 768, 8
    c1, c2, status = get_moe_cuda_config(E, M, 2 * I, H, H, I, k, "gfx950", 256, "bf16")
    assert status is True
    for c in (c1, c2):
        assert {"BLOCK_SIZE_M", "MODE", "DELTA"} <= set(c)
    assert c1["BLOCK_SIZE_M"] == c2["BLOCK_SIZE_M"] in (16, 32, 64, 128, 160)
    # an expert-parallel share: an eighth of the slots per resident expert's block choice
    e1, _, _ = get_moe_cuda_config(32, 64, 4096, 7168, 7168, 2048, 8, "gfx950", 256, "bf16", is_ep=True, ep_size=8)
    assert e1["BLOCK_SIZE_M"] == 16
    with pytest.raises(AssertionError):
        get_moe_cuda_config(E, M, 2 * I, H, H + 128, I, k, "gfx950", 256, "bf16")


# ------------------------------------------------------------------ workloads --

def test_routing_generators():
    from lightop_amd import workloads as wl

    x, w, ids = wl.make_inputs(wl.QWEN3_30B, 33, seed=1)
    assert x.shape == (33, 2048) and x.dtype == torch.bfloat16 and ids.dtype == torch.int32
    assert torch.allclose(w.sum(-1), torch.ones(33), atol=1e-5)
    assert all(len(set(r)) == 8 for r in ids.tolist()) and ids.max() < 128
    x, w, ids = wl.make_inputs(wl.DSV3_EP, 50, seed=1)
    assert torch.allclose(w.sum(-1), torch.full((50,), 2.5), atol=1e-4)
    groups = (ids // 32)
    assert all(len(set(r)) <= 4 for r in groups.tolist())       # top-4 of 8 groups
    emap = wl.expert_map_for(wl.DSV3_EP)
    assert emap[:32].tolist() == list(range(32)) and (emap[32:] == -1).all()
    assert wl.expert_map_for(wl.QWEN3_30B) is None
    # Zipf skew: the most loaded expert gets far more than the mean
    _, _, idz = wl.make_inputs(wl.DSV3_FULL, 2048, seed=0)
    counts = torch.bincount(idz.reshape(-1).long(), minlength=256)
    assert counts.max() > 4 * counts.float().mean()
    ops, nbytes, sloc, eact = wl.algorithmic_work(wl.DSV3_EP, ids, emap)
    assert ops == 6 * sloc * 2048 * 7168 and eact <= 32
    assert nbytes >= eact * 3 * 2048 * 7168


def test_weight_generator_ranges():
    from lightop_amd import workloads as wl

    w1, w2, s1, s2 = wl.make_weights(wl.TINY, seed=0)
    assert w1.shape == (8, 1024, 1024) and w2.shape == (8, 1024, 512) and s1.shape == (8, 8, 8) and s2.shape == (8, 8, 4)
    assert w1.min() >= -127 and w1.max() <= 127 and (s1 > 0).all()
    assert abs(float(torch.log(s1).mean()) - np.log(1e-3)) < 0.1


# --------------------------------------------------------------------- golden --

def _t(a, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(a))
    return t.view(torch.bfloat16) if dtype == "bf16" else t


def load_small_layer():
    z = np.load(os.path.join(GOLDEN, "small_layer.npz"))
    bf = {"x", "shared_output", "ref_c1", "ref_act", "ref_c3", "ref_out"}
    return {k: _t(z[k], "bf16" if k in bf else None) for k in z.files}


def test_golden_small_layer_oracle(oracle):
    g = load_small_layer()
    r = oracle.fused_experts_block_int8(g["x"], g["w1"], g["w2"], g["w1_scale"], g["w2_scale"], g["topk_weights"],
                                        g["topk_ids"], 16, global_num_experts=8, expert_map=g["expert_map"],
                                        routed_scaling_factor=2.5, shared_output=g["shared_output"],
                                        return_intermediates=True)
    for k, v in r.items():
        ref = g["ref_" + k]
        same = torch.equal(v.view(torch.int16), ref.view(torch.int16)) if v.dtype == torch.bfloat16 else torch.equal(v, ref)
        assert same, k


def test_golden_tiny_config1_oracle(oracle):
    from lightop_amd import workloads as wl

    doc = json.load(open(os.path.join(GOLDEN, "tiny_config1.json")))
    w1, w2, w1s, w2s = wl.make_weights(wl.TINY, seed=0)
    x, tw, ids = wl.make_inputs(wl.TINY, 64, seed=0)

    def sha(t):
        a = t.contiguous().view(torch.int16).numpy() if t.dtype == torch.bfloat16 else t.contiguous().numpy()
        return hashlib.sha256(a.tobytes()).hexdigest()

    assert {"x": sha(x), "w1": sha(w1), "topk_ids": sha(ids)}.items() <= doc["inputs_sha256"].items(), \
        "the workload generator no longer reproduces the fixture's inputs"
    r = oracle.fused_experts_block_int8(x, w1, w2, w1s, w2s, tw, ids, 16, return_intermediates=True)
    P = doc["num_tokens_post_pad"]
    assert r["num_tokens_post_pad"].item() == P
    assert r["sorted_ids"][:P].tolist() == doc["sorted_token_ids"]
    assert r["expert_ids"][: P // 16].tolist() == doc["expert_ids"]
    for k, h in doc["sha256"].items():
        assert sha(r[k]) == h, k
    # the order without fp fusion: its digests differ from the default's in c1, act and c3 on this input
    with oracle.scale_order("separate"):
        rs = oracle.fused_experts_block_int8(x, w1, w2, w1s, w2s, tw, ids, 16, return_intermediates=True)
    for k, h in doc["sha256_separate_order"].items():
        assert sha(rs[k]) == h, k
    assert any(doc["sha256_separate_order"][k] != doc["sha256"][k] for k in doc["sha256_separate_order"])


@pytest.mark.parametrize("form", ["channel", "w4a8"])
def test_golden_tiny_forms_oracle(oracle, form):
    """The per-channel and W4A8 forms of the tiny layer: the oracle still produces the committed digests."""
    from lightop_amd import workloads as wl

    doc = json.load(open(os.path.join(GOLDEN, "tiny_forms.json")))[form]
    layer, fn = {"channel": (wl.TINY_PC, oracle.fused_experts_channel_int8),
                 "w4a8": (wl.TINY_W4, oracle.fused_experts_w4a8)}[form]
    w1, w2, w1s, w2s = wl.make_weights(layer, seed=0)
    x, tw, ids = wl.make_inputs(layer, 64, seed=0)

    def sha(t):
        a = t.contiguous().view(torch.int16).numpy() if t.dtype == torch.bfloat16 else t.contiguous().numpy()
        return hashlib.sha256(a.tobytes()).hexdigest()

    assert {"x": sha(x), "w1": sha(w1), "w1_scale": sha(w1s), "topk_ids": sha(ids)}.items() \
        <= doc["inputs_sha256"].items(), "the workload generator no longer reproduces the fixture's inputs"
    r = fn(x, w1, w2, w1s, w2s, tw, ids, 16, return_intermediates=True)
    for k, h in doc["sha256"].items():
        assert sha(r[k]) == h, k
    with oracle.scale_order("separate"):  # the per-channel form scales once, at the end: no order to choose
        rs = fn(x, w1, w2, w1s, w2s, tw, ids, 16, return_intermediates=True)
    for k, h in doc.get("sha256_separate_order", {k: doc["sha256"][k] for k in ("c1", "c3", "out")}).items():
        assert sha(rs[k]) == h, k


def test_golden_align_docstring(oracle):
    doc = json.load(open(os.path.join(GOLDEN, "align_docstring.json")))
    s, e, p = oracle.moe_align_block_size(torch.tensor(doc["topk_ids"], dtype=torch.int32), doc["block_size"],
                                          doc["num_experts"])
    assert p.item() == doc["num_tokens_post_pad"]
    assert s[: p.item()].tolist() == doc["sorted_token_ids"] and e[:4].tolist() == doc["expert_ids"]


def test_torch_restatement_agrees_with_oracle_on_config1(oracle):
    """The timed CPU baseline (oracle/torch_ref.py) and the C oracle are independent
    restatements; on the tiny benchmark configuration they agree within the path's tolerance."""
    from lightop_amd import workloads as wl
    from oracle import torch_ref

    w1, w2, w1s, w2s = wl.make_weights(wl.TINY, seed=0)
    x, tw, ids = wl.make_inputs(wl.TINY, 64, seed=0)
    out = oracle.fused_experts_block_int8(x, w1, w2, w1s, w2s, tw, ids, 16).float()
    ref = torch_ref.torch_w8a8_block_int8_moe(x, w1, w2, w1s, w2s, tw, ids).float()
    err = (out - ref).abs()
    assert err.max() <= 1e-2 * ref.abs().max()
    assert err.sum() / ref.abs().sum() <= 2e-3 * 3


def test_moe_cache_is_keyed_and_grows(monkeypatch):
    """get_moe_cache hands out one buffer per (device, dtype), large enough for the call at hand:
    a later call with another dtype or a larger layer must not receive the first call's tensor
    (the reference's singleton does, fused_moe_cache.py:19-24)."""
    import torch

    from lightop_amd.moe import cache

    monkeypatch.setenv("LMSLIM_FUSED_MOE_CHUNK_SIZE", "4")
    cache.release_moe_cache()
    a = cache.get_moe_cache(2, 256, 128, "cpu", torch.bfloat16)
    assert a.dtype == torch.bfloat16 and a.dim() == 1 and a.numel() == 4 * 2 * 256
    assert cache.get_moe_cache(2, 128, 256, "cpu", torch.bfloat16) is a          # same need: shared
    assert cache.get_moe_cache(1, 64, 64, "cpu", torch.bfloat16) is a            # smaller need: shared
    b = cache.get_moe_cache(2, 256, 128, "cpu", torch.float16)
    assert b.dtype == torch.float16 and b is not a                               # another dtype: its own buffer
    c = cache.get_moe_cache(8, 512, 128, "cpu", torch.bfloat16)
    assert c.numel() == 4 * 8 * 512 and c is not a                               # larger need: grows
    assert cache.get_moe_cache(2, 256, 128, "cpu", torch.bfloat16) is c
    assert cache.moe_cache_singleton is c
    cache.release_moe_cache()
    assert cache.moe_cache_singleton is None


def test_lightop_is_an_importable_name():
    """A caller of the reference keeps its imports: the ``lightop`` package's modules are the modules of
    ``lightop_amd`` themselves (reference import paths: python/lightop/moe/__init__.py:57-78,
    python/lightop/quant/int8.py, python/lightop/gemmopt.py:437, python/lightop/moe_fused_gate.py:10)."""
    import lightop
    import lightop_amd
    from lightop.moe import fused_experts_impl_int8, fused_experts_impl_w4a8, moe_align_block_size, moe_sum, topk_softmax
    from lightop.moe.native import fused_experts_impl_int8 as native_entry
    from lightop.quant import per_token_group_quant_int8, per_token_quant_int8
    from lightop.quant.int8 import per_token_group_quant_int8 as q2
    from lightop.gemmopt import moe_gemm_w8a8
    from lightop.moe_fused_gate import moe_fused_gate
    from lightop.fuse_silu_mul_quant import fuse_silu_mul_quant as fsq
    from lightop import envs, fuse_silu_mul_quant, op

    assert lightop.moe is lightop_amd.moe and lightop.quant is lightop_amd.quant and op is lightop_amd.op
    assert fused_experts_impl_int8 is lightop_amd.moe.fused_experts_impl_int8 is native_entry
    assert fused_experts_impl_w4a8 is lightop_amd.moe.fused_experts_impl_w4a8
    assert moe_align_block_size is lightop_amd.moe.moe_align_block_size and moe_sum is lightop_amd.moe.moe_sum
    assert topk_softmax is lightop_amd.op.topk_softmax and moe_fused_gate is lightop_amd.moe.moe_fused_gate
    assert per_token_group_quant_int8 is q2 is lightop_amd.quant.per_token_group_quant_int8
    assert per_token_quant_int8 is lightop_amd.quant.per_token_quant_int8
    assert moe_gemm_w8a8 is lightop_amd.gemmopt.moe_gemm_w8a8 is lightop_amd.moe.moe_gemm_w8a8
    assert fuse_silu_mul_quant is fsq is lightop_amd.fuse_silu_mul_quant  # the function, as in the reference
    assert envs.LMSLIM_FUSED_MOE_CHUNK_SIZE == lightop_amd.envs.LMSLIM_FUSED_MOE_CHUNK_SIZE
    with pytest.raises(AttributeError):  # an operator family outside the path
        lightop.RMSNorm
    with pytest.raises(AttributeError):
        lightop.moe.fused_experts_impl_fp8_marlin
    import lightop.quant.int8 as q8  # the attribute form of the dotted import
    import lightop_amd.quant as q

    assert q8 is q and q.int8 is q


def test_tuning_files_override_the_compiled_table(monkeypatch, tmp_path):
    """TRITON_JSON_DIR (vllm_compat/w8a8_get_cache_json.py:24) names a directory of tuning files in the
    reference's layout; the block size such a file holds for the nearest tuned token count comes back from
    get_w8a8moe_json (reference lookup: int8.py:220-256) together with the kernel that size launches."""
    from lightop_amd import _lib, moe
    from lightop_amd.moe import tile_files

    E, k, H, I = 128, 8, 2048, 768
    monkeypatch.delenv("TRITON_JSON_DIR", raising=False)
    tile_files.forget()
    c1, c2 = moe.get_w8a8moe_json(8192, E, 2 * I, H, I, True, [128, 128], k)
    assert (c1["BLOCK_SIZE_M"], c1["source"], c1["kernel"]) == (128, "compiled", _lib.LO_KERNEL_T128)
    assert tile_files.block_size_m(8192, E, 2 * I, H, I, k, [128, 128]) == 0

    cfg = lambda bs, **kw: dict({"BLOCK_SIZE_M": bs, "BLOCK_SIZE_N": 256, "BLOCK_SIZE_K": 128, "GROUP_SIZE_M": 1,
                                 "num_warps": 4, "num_stages": 0}, **kw)
    table = {"1": {"config1": cfg(16, lightop_amd_two_launch=True), "config2": cfg(16, lightop_amd_two_launch=True)},
             "64": {"config1": cfg(32), "config2": cfg(32)},
             "8192": {"config1": cfg(64), "config2": cfg(64)}}
    name = tile_files.file_name(E, 2 * I, H, I, k, [128, 128], False)
    assert name == "MOE_BLOCKINT8[128,128]_E=128_N1=1536_N2=2048_K=768_TOPK8_gfx950_256cu.json"
    with open(tmp_path / name, "w") as f:
        json.dump({f"{2 * I}_{H}_{I}": table}, f)
    monkeypatch.setenv("TRITON_JSON_DIR", str(tmp_path))
    tile_files.forget()
    c1, c2 = moe.get_w8a8moe_json(8192, E, 2 * I, H, I, True, [128, 128], k)
    assert (c1["BLOCK_SIZE_M"], c2["BLOCK_SIZE_M"], c1["source"]) == (64, 64, "file")
    assert c1["kernel"] == _lib.LO_KERNEL_TILE           # the kernel that block size launches, not the table's
    # nearest tuned count on a logarithmic scale: 3000 -> 8192, 500 -> 64 (a factor 7.8 away, 8192 is 16.4), 40 -> 64
    assert tile_files.block_size_m(3000, E, 2 * I, H, I, k, [128, 128]) == 64
    assert tile_files.block_size_m(500, E, 2 * I, H, I, k, [128, 128]) == 32
    assert tile_files.block_size_m(40, E, 2 * I, H, I, k, [128, 128]) == 32
    # the tuner's mark "the library's own pick was fastest" (the two-launch path): nothing is forced
    assert tile_files.block_size_m(2, E, 2 * I, H, I, k, [128, 128]) == 0
    c1, _ = moe.get_w8a8moe_json(1, E, 2 * I, H, I, True, [128, 128], k)
    assert (c1["kernel"], c1["source"]) == (_lib.LO_KERNEL_DEC, "compiled")
    # another layer shape has no file: the compiled-in table answers
    c1, _ = moe.get_w8a8moe_json(8192, 32, 4096, 7168, 2048, True, [128, 128], k, global_num_experts=256)
    assert (c1["BLOCK_SIZE_M"], c1["source"]) == (128, "compiled")
    # per-channel and int4 forms have file names of their own (w8a8_get_cache_json.py:133-149)
    assert tile_files.file_name(8, 1024, 1024, 512, 2, None, False).startswith("MOE_W8A8INT8_E=8_")
    assert tile_files.file_name(8, 1024, 1024, 512, 2, [1, 128], True).startswith("MOE_W4A8INT8[1,128]_E=8_")
    assert tile_files.file_name(8, 1024, 1024, 512, 2, None, True).startswith("MOE_W4A8INT8_E=8_")
    # 160-token blocks of int4 weights: a file's entry is used where the call can take it, and left to the table where it cannot
    name = tile_files.file_name(E, 2 * I, H, I, k, [1, 128], True)
    with open(tmp_path / name, "w") as f:
        json.dump({f"{2 * I}_{H}_{I}": {"1900": {"config1": cfg(160), "config2": cfg(160)}}}, f)
    w4 = lambda m=1900, **kw: moe.get_w8a8moe_json(m, E, 2 * I, H, I, True, [1, 128], k, int4=True, **kw)[0]
    assert (w4()["BLOCK_SIZE_M"], w4()["kernel"], w4()["source"]) == (160, _lib.LO_KERNEL_T128, "file")
    for kw in ({"dtype": torch.float16}, {"activation": "gelu"}, {"m": 2500}):
        assert (w4(**kw)["BLOCK_SIZE_M"], w4(**kw)["source"]) == (128, "compiled")
    monkeypatch.delenv("TRITON_JSON_DIR")
    tile_files.forget()


def test_expert_ids_must_cover_the_blocks_the_grid_reaches():
    """The GEMM stubs refuse an expert_ids tensor shorter than the token blocks sorted_token_ids has room for
    (the kernels may read any such block's entry before they know how many blocks are in use)."""
    import pytest
    import torch

    from lightop_amd.moe.native import _check_block_extents

    sorted_ids = torch.zeros(128 * 7 + 5, dtype=torch.int32)
    _check_block_extents(sorted_ids, torch.zeros(7, dtype=torch.int32), 128, 10_000)   # 7 whole blocks
    _check_block_extents(sorted_ids, torch.zeros(3, dtype=torch.int32), 128, 3)        # at most one block per slot
    with pytest.raises(ValueError, match="span 7 blocks"):
        _check_block_extents(sorted_ids, torch.zeros(6, dtype=torch.int32), 128, 10_000)


@pytest.mark.parametrize("problem", ["another torch", "older binding", "missing"])
def test_calls_go_through_python_without_a_usable_binding(problem, monkeypatch):
    """A host binding that is missing, or built for another torch, is not used: one warning, and every call is declined,
    so that Python marshals it."""
    import sys

    import lightop_amd
    from lightop_amd import _lib

    monkeypatch.setattr(_lib, "_host", None)
    if problem == "missing":
        monkeypatch.setitem(sys.modules, "lightop_amd._host", None)
        monkeypatch.delattr(lightop_amd, "_host", raising=False)
    else:
        from lightop_amd import _host

        assert _host.built_for == _lib.binding_key()  # the one that is there is this torch's
        if problem == "another torch":
            monkeypatch.setattr(_host, "built_for", "torch 2.9.1+rocm6.4, Python 3.10")
        else:
            monkeypatch.delattr(_host, "built_for")
    with pytest.warns(RuntimeWarning, match="host binding"):
        host = _lib.host()
    assert _lib.host() is host
    assert host.topk_softmax(*range(5)) is None and host.fused_gate(*range(9)) is None and host.fused_experts(*range(16)) is None
