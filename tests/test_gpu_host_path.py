"""The native marshalling of the whole-path call and of the routers (csrc/host_binding.cpp) against the Python
marshalling beside it, bit for bit: the ordinary calls it takes, and the ones it has to leave to Python."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _layer(form, dev):
    from lightop_amd import workloads as wl
    from lightop_amd.moe import preshuffle_moe_scale_int4, preshuffle_moe_weight, preshuffle_moe_weight_int4

    layer = {"rows": wl.TINY, "block": wl.TINY, "channel": wl.TINY_PC, "w4": wl.TINY_W4, "w4_channel": wl.TINY_W4_PC}[form]
    w1, w2, w1s, w2s = wl.make_weights(layer, seed=0, device=dev)
    if form == "block":
        w1, w2 = preshuffle_moe_weight(w1), preshuffle_moe_weight(w2)
    elif form.startswith("w4"):
        w1, w2 = preshuffle_moe_weight_int4(w1), preshuffle_moe_weight_int4(w2)
        if form == "w4":
            w1s, w2s = preshuffle_moe_scale_int4(w1s), preshuffle_moe_scale_int4(w2s)
    return layer, (w1, w2), {"w1_scale": w1s, "w2_scale": w2s}


@pytest.mark.parametrize("variant", ["plain", "int64 ids", "share", "inplace", "strided ids", "chunks", "other stream"])
@pytest.mark.parametrize("form", ["rows", "block", "channel", "w4", "w4_channel"])
def test_whole_path(form, variant, monkeypatch):
    from lightop_amd import _lib, workloads as wl
    from lightop_amd.moe import fused_experts_impl_int8, fused_experts_impl_w4a8

    dev = torch.device("cuda:0")
    print(f"[case] host path {form} {variant}", flush=True)
    layer, weights, kw = _layer(form, dev)
    M = 37
    x, tw, ids = (t.to(dev) for t in wl.make_inputs(layer, M, seed=3))
    cache13 = torch.empty(M * layer.top_k * max(2 * layer.I, layer.H), dtype=torch.bfloat16, device=dev)
    if form.startswith("w4"):
        fn, kw["block_shape"] = fused_experts_impl_w4a8, [1, 128] if form == "w4" else None
    else:
        fn, kw["block_shape"] = fused_experts_impl_int8, None if form == "channel" else [128, 128]
        kw.update(use_int8_w8a8=True, per_channel_quant=form == "channel")
    if variant == "int64 ids":
        ids = ids.long()
    elif variant == "strided ids":  # a conversion to make: left to Python
        ids = torch.stack([ids, ids], dim=-1)[..., 0]
    elif variant == "chunks":       # three chunks: left to Python
        monkeypatch.setenv("LMSLIM_FUSED_MOE_CHUNK_SIZE", "16")
    elif variant == "share":
        emap = torch.full((2 * layer.E,), -1, dtype=torch.int32, device=dev)
        emap[1::2] = torch.arange(layer.E, dtype=torch.int32, device=dev)
        ids = ids * 2 + (ids + torch.arange(M, device=dev, dtype=torch.int32)[:, None]) % 2
        kw.update(expert_map=emap, global_num_experts=2 * layer.E, routed_scaling_factor=2.5, shared_output=x + 1)

    ws = torch.empty(64 << 20, dtype=torch.uint8, device=dev)
    want = fn(x.clone(), *weights, tw, ids, cache13, lightop_amd_workspace=ws, **kw)  # a private knob: Python's marshalling
    xin = x.clone()
    if variant == "other stream":
        torch.cuda.synchronize()
        with torch.cuda.stream(torch.cuda.Stream()):
            got = fn(xin, *weights, tw, ids, cache13, **kw)
    else:
        got = fn(xin, *weights, tw, ids, cache13, inplace=variant == "inplace", **kw)
    torch.cuda.synchronize()
    assert (got.data_ptr() == xin.data_ptr()) == (variant == "inplace")
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))

    # which of the two marshalled it
    form_no = {"rows": 0, "block": 0, "channel": 1, "w4": 2, "w4_channel": 3}[form]
    direct = _lib.host().fused_experts(x, *weights, tw, ids, cache13, kw["w1_scale"], kw["w2_scale"], kw.get("expert_map"),
                                       kw.get("shared_output"), form_no, False, False, kw.get("global_num_experts", -1),
                                       kw.get("routed_scaling_factor", 1.0), 0)
    assert (direct is None) == (variant in ("strided ids", "chunks"))
    if direct is not None:
        assert torch.equal(direct.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("renorm", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_routers(dtype, renorm):
    """Both marshallings write the same outputs; arguments the native one declines are still refused."""
    from lightop_amd import _lib
    from lightop_amd.moe import moe_fused_gate, topk_softmax

    dev, T, E, k = torch.device("cuda:0"), 19, 64, 6
    g = torch.randn(T, E, device=dev).to(dtype)
    outs = []
    for native in (True, False):
        w, i = torch.zeros(T, k, device=dev), torch.zeros(T, k, dtype=torch.int64, device=dev)
        src = torch.zeros(T, k, dtype=torch.int32, device=dev)
        if native:
            assert _lib.host().topk_softmax(w, i, src, g, renorm) is True
        else:
            _lib.check(_lib.lib().lo_topk_softmax(_lib.ptr(g), {torch.float32: 2, torch.bfloat16: 0}[dtype], T, E, k, int(renorm),
                                                  _lib.ptr(w), _lib.ptr(i), _lib.LO_I64, _lib.ptr(src), _lib.stream_of(g)))
        outs.append((w, i, src))
    assert all(torch.equal(a, b) for a, b in zip(*outs))
    bias = torch.randn(E, device=dev)
    w, i = moe_fused_gate(g, bias, 8, 4, k, 0, 2.5)
    assert w.dtype == torch.float32 and i.dtype == torch.int32 and w.shape == i.shape == (T, k)
    with pytest.raises(RuntimeError, match="contiguous"):
        topk_softmax(torch.empty(T, k, device=dev), torch.empty(T, k, dtype=torch.int32, device=dev), None, g.t(), renorm)
    with pytest.raises(RuntimeError, match="GPU"):
        moe_fused_gate(g, bias.cpu(), 8, 4, k, 0, 2.5)
    with pytest.raises(RuntimeError, match="topk_group"):
        moe_fused_gate(g, bias, 8, 9, k, 0, 2.5)


@pytest.mark.parametrize("warm", [False, True])
def test_out_of_memory_keeps_its_type(warm):
    """A call whose output or workspace does not fit raises torch's own out-of-memory error, as the allocation in Python
    does, and works again once there is room.  ``warm``: the stream has a smaller workspace that has to grow."""
    from lightop_amd import workloads as wl
    from lightop_amd.moe import fused_experts_impl_int8

    dev, M = torch.device("cuda:0"), 16384
    print(f"[case] out of memory warm={warm}", flush=True)
    layer, weights, kw = _layer("block", dev)
    x, tw, ids = (t.to(dev) for t in wl.make_inputs(layer, M, seed=3))
    cache13 = torch.empty(M * layer.top_k * max(2 * layer.I, layer.H), dtype=torch.bfloat16, device=dev)

    def run(m, inplace):
        return fused_experts_impl_int8(x[:m].clone() if inplace else x[:m], *weights, tw[:m], ids[:m], cache13, inplace=inplace,
                                       use_int8_w8a8=True, block_shape=[128, 128], **kw)

    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        if warm:
            run(64, False)
        held = x.clone()  # what an in-place call works on
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        total = torch.cuda.get_device_properties(dev).total_memory
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (1 << 20)) / total)
        try:
            with pytest.raises(torch.cuda.OutOfMemoryError):
                run(M, False)
            with pytest.raises(torch.cuda.OutOfMemoryError):  # the workspace alone
                fused_experts_impl_int8(held, *weights, tw, ids, cache13, inplace=True, use_int8_w8a8=True,
                                        block_shape=[128, 128], **kw)
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        assert torch.equal(held, x)
        got = run(M, False)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), run(M, True).view(torch.int16))
