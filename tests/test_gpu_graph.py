"""The whole path recorded into a HIP graph: every replay must reproduce the eager result.

The C entry points allocate nothing and never synchronise, and what the Python ones allocate under a capture lives as long
as the graph, so a caller may capture them.
The replays are separated by eager work and synchronisations of the program itself."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 16, 64])
@pytest.mark.parametrize("form", ["block", "block_preshuffled", "channel", "w4"])
def test_graph_replays_match_eager(M, form):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from lightop_amd import _lib, workloads as wl
    from lightop_amd.moe import (fused_experts_impl_int8, fused_experts_impl_w4a8, preshuffle_moe_scale_int4,
                                 preshuffle_moe_weight, preshuffle_moe_weight_int4)

    _lib.lib()
    dev = torch.device("cuda:0")
    layer = {"block": wl.TINY, "block_preshuffled": wl.TINY, "channel": wl.TINY_PC, "w4": wl.TINY_W4}[form]
    w1, w2, w1s, w2s = wl.make_weights(layer, seed=0, device=dev)
    if form == "w4":
        w1, w2 = preshuffle_moe_weight_int4(w1), preshuffle_moe_weight_int4(w2)
        w1s, w2s = preshuffle_moe_scale_int4(w1s), preshuffle_moe_scale_int4(w2s)
    if form == "block_preshuffled":  # load-time layout: the two-launch path at 1 and 16 tokens
        w1, w2 = preshuffle_moe_weight(w1), preshuffle_moe_weight(w2)
    x, tw, ids = (t.to(dev) for t in wl.make_inputs(layer, M, seed=5))
    cache13 = torch.empty(M * layer.top_k * max(2 * layer.I, layer.H), dtype=torch.bfloat16, device=dev)

    def run():
        if form == "w4":
            return fused_experts_impl_w4a8(x, w1, w2, tw, ids, cache13, w1_scale=w1s, w2_scale=w2s,
                                           block_shape=[1, 128])
        return fused_experts_impl_int8(x, w1, w2, tw, ids, cache13, use_int8_w8a8=True,
                                       per_channel_quant=form == "channel", w1_scale=w1s, w2_scale=w2s,
                                       block_shape=None if form == "channel" else [128, 128])

    print(f"[case] graph replay M={M} {form}", flush=True)
    eager = run().clone()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = run()
    for rep in range(4):
        out.zero_()
        cache13.fill_(float(rep))                 # eager work between the replays
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), eager.view(torch.int16)), f"replay {rep} differs"


class HipGraph:
    """A graph recorded with the runtime's own calls on a stream of the program's, which torch's allocator does not
    know to be capturing into a graph."""

    def __init__(self, stream, fn):
        from lightop_amd import _lib

        hip = _lib.lib()  # (symbols of the HIP runtime it is linked against)
        self.hip, self.exec, graph = hip, ctypes.c_void_p(), ctypes.c_void_p()
        self.check(hip.hipStreamBeginCapture(ctypes.c_void_p(stream.cuda_stream), 2))  # relaxed
        with torch.cuda.stream(stream):
            self.out = fn()
        self.check(hip.hipStreamEndCapture(ctypes.c_void_p(stream.cuda_stream), ctypes.byref(graph)))
        self.check(hip.hipGraphInstantiate(ctypes.byref(self.exec), graph, None, None, ctypes.c_size_t(0)))

    @staticmethod
    def check(rc):
        assert rc == 0, f"HIP error {rc}"

    def replay(self):
        self.check(self.hip.hipGraphLaunch(self.exec, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))


@pytest.mark.parametrize("capture", ["torch", "torch without snapshots", "runtime"])
def test_replays_write_to_no_memory_of_others(capture, monkeypatch):
    """A graph's scratch stays the graph's: after a warm-up and a capture on one stream, larger calls there and calls on
    more streams than workspaces are kept for, the memory that stream then gets from the allocator survives replays."""
    from lightop_amd import workloads as wl
    from lightop_amd.moe import fused_experts_impl_int8, native, preshuffle_moe_weight

    dev, layer, M = torch.device("cuda:0"), wl.TINY, 48
    print(f"[case] graph scratch {capture}", flush=True)
    w1, w2, w1s, w2s = wl.make_weights(layer, seed=0, device=dev)
    w1, w2 = preshuffle_moe_weight(w1), preshuffle_moe_weight(w2)
    args = {m: tuple(t.to(dev) for t in wl.make_inputs(layer, m, seed=m)) for m in (M, 4096)}
    cache13 = torch.empty(4096 * layer.top_k * max(2 * layer.I, layer.H), dtype=torch.bfloat16, device=dev)

    def run(m=M):
        x, tw, ids = args[m]
        return fused_experts_impl_int8(x, w1, w2, tw, ids, cache13, use_int8_w8a8=True, w1_scale=w1s, w2_scale=w2s,
                                       block_shape=[128, 128])

    monkeypatch.setattr(native, "_capture_kept", {})
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        eager = run().clone()
    torch.cuda.synchronize()
    if capture == "torch without snapshots":
        def refuse():
            raise RuntimeError("snapshots are not supported")

        monkeypatch.setattr(torch.cuda, "memory_snapshot", refuse)
    if capture != "runtime":
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            out = run()
    else:
        g = HipGraph(side, run)
        out = g.out
    assert list(native._capture_kept) == ([] if capture == "torch" else [(0, side.cuda_stream)])  # torch's graphs own theirs
    torch.cuda.synchronize()
    for stream in [torch.cuda.Stream() for _ in range(20)] + [side]:
        with torch.cuda.stream(stream):
            for m in (M, 4096):
                run(m)
        torch.cuda.synchronize()
    with torch.cuda.stream(side):
        canaries = [torch.full((n,), 0x5A, dtype=torch.uint8, device=dev) for n in (1 << 20, 2 << 20, 16 << 20) for _ in range(8)]
    for rep in range(4):
        out.zero_()
        cache13.fill_(float(rep))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), eager.view(torch.int16)), f"replay {rep} differs"
        assert all(bool((c == 0x5A).all()) for c in canaries), f"replay {rep} wrote to memory of others"
