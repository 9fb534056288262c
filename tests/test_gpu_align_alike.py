"""Routing that sends many slots of a wave to one expert (rows of padding tokens alike, every token to one expert), in the
alignment by several workgroups (csrc/align.hip, moe_align_wide_body): the copies of its counters at the ends of each number of
copies, bit for bit against the CPU oracle or shorter calls, and the time that they are there for."""
import dataclasses

import pytest
import torch

pytestmark = pytest.mark.gpu


def _ids(kind, M, k, E):
    g = torch.Generator().manual_seed(M + E)
    ids = torch.rand(M, E, generator=g).topk(k, 1).indices
    if kind == "one":
        ids[:] = E - 1
    elif kind == "rows":
        ids[M // 3:] = torch.randperm(E, generator=g)[:k]
    return ids.to(torch.int32)


def _align(dev, ids, E, bs):
    from lightop_amd import op

    cap = ids.numel() + E * (bs - 1)
    s = torch.full((cap,), -7, dtype=torch.int32, device=dev)
    e = torch.full(((cap + bs - 1) // bs,), -7, dtype=torch.int32, device=dev)
    p = torch.full((1,), -7, dtype=torch.int32, device=dev)
    return lambda: op.moe_align_block_size(ids, E, bs, s, e, p), s, e, p


@pytest.mark.parametrize("M,E", [(512, 590), (512, 591), (512, 698), (512, 699), (2560, 591), (2561, 591), (4096, 100), (4097, 100),
                                 (4128, 129), (4129, 129)])
@pytest.mark.parametrize("kind", ["one", "rows"])
def test_align(oracle, M, E, kind):
    dev, bs = torch.device("cuda:0"), 64
    print(f"[case] alignment of rows alike M={M} E={E} {kind}", flush=True)
    ids = _ids(kind, M, 8, E)
    call, s, e, p = _align(dev, ids.to(dev), E, bs)
    call()
    torch.cuda.synchronize()
    rs, re, rp = oracle.moe_align_block_size(ids, bs, E)
    P = rp.item()
    assert p.item() == P
    assert torch.equal(s.cpu()[:P], rs[:P]) and bool((s.cpu()[P:] == ids.numel()).all())
    assert torch.equal(e.cpu()[: P // bs], re[: P // bs]) and bool((e.cpu()[P // bs:] == -1).all())


@pytest.mark.parametrize("M,H,k,E_global", [(2512, 7168, 8, 365), (2512, 7168, 8, 366), (2512, 7168, 8, 512), (2511, 7168, 8, 64),
                                            (5023, 3584, 5, 64), (5024, 3584, 5, 64), (8192, 5632, 8, 64), (8193, 5632, 8, 64),
                                            (2000, 1024, 4, 64), (2001, 1024, 4, 64)])
@pytest.mark.parametrize("channel", [False, True])
def test_beside_the_quantisation(M, H, k, E_global, channel):
    """Either side of the lines (values, slots, experts, slots a token), two thirds of the rows alike."""
    from lightop_amd import workloads as wl
    from lightop_amd.moe import fused_experts_impl_int8, get_moe_cache, preshuffle_moe_weight

    dev = torch.device("cuda:0")
    print(f"[case] alignment of rows alike in the whole path M={M} H={H} k={k} E={E_global} channel={channel}", flush=True)
    layer = dataclasses.replace(wl.TINY, H=H, I=128, top_k=k, E_global=E_global, quant="channel" if channel else "block")
    w1, w2, w1s, w2s = wl.make_weights(layer, seed=3, device=dev, gen_device="cuda")
    w1, w2 = preshuffle_moe_weight(w1), preshuffle_moe_weight(w2)
    g = torch.Generator(device=dev).manual_seed(M)
    x = torch.randn((M, H), generator=g, device=dev).to(torch.bfloat16)
    tw = torch.rand((M, k), generator=g, device=dev)
    ids = _ids("rows", M, k, E_global).to(dev)

    def run(rows):
        return fused_experts_impl_int8(
            x[rows], w1, w2, tw[rows], ids[rows], get_moe_cache(k, 2 * layer.I, H, dev, torch.bfloat16), use_int8_w8a8=True,
            per_channel_quant=channel, global_num_experts=E_global, expert_map=wl.expert_map_for(layer, dev), w1_scale=w1s,
            w2_scale=w2s, block_shape=None if channel else [128, 128])

    got = run(slice(0, M))
    for a in sorted({0, M // 3 // 128 * 128, (M - 1) // 128 * 128}):
        rows = slice(a, min(a + 128, M))
        assert torch.equal(got[rows].view(torch.int16), run(rows).view(torch.int16))


def _us(call):
    """Launches alone, from a graph of ten calls."""
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(10):
            call()
    times = []
    for _ in range(9):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        graph.replay()
        b.record()
        torch.cuda.synchronize()
        times.append(a.elapsed_time(b) * 100)
    return sorted(times)[4]


def test_one_expert_costs_no_multiple_of_spread_routing():
    """32768 slots, 128 experts: 19.5 us with every slot on one expert, 10.2 spread; with one counter an expert and workgroup 32.6
    and 9.8."""
    dev = torch.device("cuda:0")
    print("[case] time of the alignment of 32768 slots on one of 128 experts", flush=True)
    us = {kind: _us(_align(dev, _ids(kind, 4096, 8, 128).to(dev), 128, 64)[0]) for kind in ("spread", "one")}
    assert us["one"] < 2.6 * us["spread"], us


@pytest.mark.parametrize("M,E", [(5000, 100), (5000, 600)])
def test_without_scratch(oracle, M, E):
    """Past the lines that the counters' own launch draws, a call that brings no memory for them is aligned by several workgroups all
    the same: about as fast as with it, where one workgroup takes more than twice as long (600 experts 53 us, 24.5 with)."""
    from lightop_amd import _lib

    dev, bs = torch.device("cuda:0"), 64
    print(f"[case] alignment without scratch M={M} E={E}", flush=True)
    ids = _ids("rows", M, 8, E)
    with_scratch, s, e, p = _align(dev, ids.to(dev), E, bs)
    on_gpu = ids.to(dev)

    def without():
        _lib.check(_lib.lib().lo_moe_align_block_size(
            _lib.ptr(on_gpu), _lib.LO_I32, on_gpu.numel(), E, bs, None, 0, _lib.ptr(s), s.numel(), _lib.ptr(e), e.numel(),
            _lib.ptr(p), _lib.stream_of(on_gpu)))

    without()
    torch.cuda.synchronize()
    rs, re, rp = oracle.moe_align_block_size(ids, bs, E)
    P = rp.item()
    assert p.item() == P and torch.equal(s.cpu()[:P], rs[:P]) and torch.equal(e.cpu()[: P // bs], re[: P // bs])
    us = _us(without), _us(with_scratch)
    assert us[0] < 2.0 * us[1], us
