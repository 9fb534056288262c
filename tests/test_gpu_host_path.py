"""The native marshalling of the whole-path call and of the routers (csrc/host_binding.cpp) against the Python
marshalling beside it, bit for bit: the ordinary calls it takes, and the ones it has to leave to Python; threads and errors."""
import ctypes
import subprocess
import threading
import time

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


STUB = """
#include <unistd.h>
volatile int entered, let_go;
int stub(void) {
  entered = 1;
  for (int i = 0; i < 5000 && !let_go; ++i) usleep(1000);
  return let_go ? 0 : -1;
}
const char *message(void) { return "no other thread ran during the call"; }
"""


@pytest.mark.parametrize("entry", ["block", "channel", "topk_softmax", "fused_gate"])
def test_other_threads_run_during_a_launch(entry, tmp_path):
    """A launch may wait (for room in the queue, for a table), and what it waits for may need the interpreter: in the place
    of the library's function, one that returns when another Python thread has run, or after five seconds."""
    from lightop_amd import _lib, workloads as wl

    dev = torch.device("cuda:0")
    print(f"[case] threads during a launch {entry}", flush=True)
    (tmp_path / "stub.c").write_text(STUB)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(tmp_path / "stub.so"), str(tmp_path / "stub.c")], check=True)
    stub = ctypes.CDLL(str(tmp_path / "stub.so"))
    entered, let_go = ctypes.c_int.in_dll(stub, "entered"), ctypes.c_int.in_dll(stub, "let_go")
    layer, weights, kw = _layer("channel" if entry == "channel" else "block", dev)
    x, tw, ids = (t.to(dev) for t in wl.make_inputs(layer, 4, seed=3))
    cache13 = torch.empty(4 * layer.top_k * max(2 * layer.I, layer.H), dtype=torch.bfloat16, device=dev)
    g, bias = torch.randn(4, 64, device=dev), torch.zeros(64, device=dev)

    def other():
        for _ in range(20000):
            if entered.value:
                let_go.value = 1
                return
            time.sleep(0.0005)

    host, real = _lib.host(), _lib.lib()
    address = lambda fn: ctypes.cast(fn, ctypes.c_void_p).value  # noqa: E731
    thread = threading.Thread(target=other)
    thread.start()
    try:
        host.bind(*[address(stub.stub)] * 2, address(real.lo_fused_experts_workspace_bytes), *[address(stub.stub)] * 2,
                  address(stub.message))
        if entry == "topk_softmax":
            out = host.topk_softmax(torch.empty(4, 6, device=dev), torch.empty(4, 6, dtype=torch.int32, device=dev), None, g, True)
        elif entry == "fused_gate":
            out = host.fused_gate(g, bias, 8, 4, 6, 0, 2.5, False, False)
        else:
            out = host.fused_experts(x, *weights, tw, ids, cache13, kw["w1_scale"], kw["w2_scale"], None, None,
                                     int(entry == "channel"), False, False, -1, 1.0, 0)
        assert out is not None and let_go.value == 1
    finally:
        _lib._host = None
        _lib.host()  # the library's own functions again
        thread.join()


ALLOCATOR = """
#include <stddef.h>
#include <sys/types.h>
#include <unistd.h>
int (*real_malloc)(void **, size_t);
int (*real_free)(void *);
volatile int entered, let_go, waited_in_vain;
void *take(ssize_t bytes, int device, void *stream) {
  void *p = NULL;
  entered = 1;
  for (int i = 0; i < 5000 && !let_go; ++i) usleep(1000);
  waited_in_vain |= !let_go;
  return real_malloc(&p, (size_t)bytes) ? NULL : p;
}
void give(void *p, ssize_t bytes, int device, void *stream) { real_free(p); }
"""


@pytest.mark.parametrize("entry", ["block", "fused_gate"])
def test_other_threads_run_during_an_allocation(entry, tmp_path):
    """Short of memory an allocation waits for the GPU, and what that waits for may need the interpreter: outputs come from
    an allocator that returns when another Python thread has run, or after five seconds."""
    from lightop_amd import _lib, workloads as wl

    dev = torch.device("cuda:0")
    print(f"[case] threads during an allocation {entry}", flush=True)
    (tmp_path / "stub.c").write_text(ALLOCATOR)
    path = str(tmp_path / "stub.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", path, str(tmp_path / "stub.c")], check=True)
    stub, host, hip = ctypes.CDLL(path), _lib.host(), _lib.lib()
    for name, fn in (("real_malloc", hip.hipMalloc), ("real_free", hip.hipFree)):
        ctypes.c_void_p.in_dll(stub, name).value = ctypes.cast(fn, ctypes.c_void_p).value
    entered, let_go, in_vain = (ctypes.c_int.in_dll(stub, n) for n in ("entered", "let_go", "waited_in_vain"))
    layer, weights, kw = _layer("block", dev)
    x, tw, ids = (t.to(dev) for t in wl.make_inputs(layer, 4, seed=3))
    cache13 = torch.empty(4 * layer.top_k * max(2 * layer.I, layer.H), dtype=torch.bfloat16, device=dev)
    g, bias = torch.randn(4, 64, device=dev), torch.zeros(64, device=dev)

    def call():
        if entry == "fused_gate":
            return host.fused_gate(g, bias, 8, 4, 6, 0, 2.5, False, False)[0]
        return host.fused_experts(x, *weights, tw, ids, cache13, kw["w1_scale"], kw["w2_scale"], None, None, 0, False, False, -1,
                                  1.0, 0)

    def other():
        for _ in range(20000):
            if entered.value:
                let_go.value = 1
                return
            time.sleep(0.0005)

    want = call()  # (the workspace is there from now on)
    allocator = torch.cuda.memory.CUDAPluggableAllocator(path, "take", "give")
    pool = torch.cuda.MemPool(allocator.allocator())
    thread = threading.Thread(target=other)
    thread.start()
    try:
        with torch.cuda.use_mem_pool(pool):
            got = call()
    finally:
        entered.value = 1
        thread.join()
    torch.cuda.synchronize()
    same = torch.equal(got, want)
    del got, pool  # the pool gives its memory back through the allocator, which it does not keep alive
    assert same and not in_vain.value


@pytest.mark.parametrize("form", ["block", "channel"])
def test_threads_share_a_stream(form):
    """Two threads that queue calls of different sizes on one stream: neither's launches come between the other's, whose
    intermediates are in the same workspace."""
    from lightop_amd import workloads as wl
    from lightop_amd.moe import fused_experts_impl_int8

    dev = torch.device("cuda:0")
    print(f"[case] threads on one stream {form}", flush=True)
    layer, weights, kw = _layer(form, dev)
    kw.update(use_int8_w8a8=True, per_channel_quant=form == "channel", block_shape=None if form == "channel" else [128, 128])
    sizes = (300, 77)
    inputs = [tuple(t.to(dev) for t in wl.make_inputs(layer, m, seed=m)) for m in sizes]
    caches = [torch.empty(m * layer.top_k * max(2 * layer.I, layer.H), dtype=torch.bfloat16, device=dev) for m in sizes]

    def call(i):
        x, tw, ids = inputs[i]
        return fused_experts_impl_int8(x, *weights, tw, ids, caches[i], **kw)

    want = [call(i).clone() for i in (0, 1)]
    torch.cuda.synchronize()
    got = [[], []]
    threads = [threading.Thread(target=lambda i=i: got[i].extend(call(i) for _ in range(200))) for i in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for i in (0, 1):
        assert len(got[i]) == 200 and all(torch.equal(o.view(torch.int16), want[i].view(torch.int16)) for o in got[i])


def test_without_the_binding(monkeypatch):
    """The routers and the whole path with the Python marshalling alone."""
    from lightop_amd import _lib, workloads as wl
    from lightop_amd.moe import fused_experts_impl_int8, moe_fused_gate, topk_softmax

    dev = torch.device("cuda:0")
    layer, weights, kw = _layer("block", dev)
    x, _, _ = (t.to(dev) for t in wl.make_inputs(layer, 21, seed=3))
    logits = torch.randn(21, layer.E, device=dev)
    cache13 = torch.empty(21 * layer.top_k * max(2 * layer.I, layer.H), dtype=torch.bfloat16, device=dev)
    outs = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(_lib, "_host", _lib._NoHost())
        w, ids = torch.empty(21, layer.top_k, device=dev), torch.empty(21, layer.top_k, dtype=torch.int32, device=dev)
        topk_softmax(w, ids, None, logits, True)
        gw, gi = moe_fused_gate(logits, torch.zeros(layer.E, device=dev), 2, 1, 2, 0, 2.5)
        out = fused_experts_impl_int8(x, *weights, w, ids, cache13, use_int8_w8a8=True, block_shape=[128, 128], **kw)
        outs.append((w, ids, gw, gi, out.view(torch.int16)))
    assert all(torch.equal(a, b) for a, b in zip(*outs))
