"""The alignment by several workgroups in one launch (csrc/align.hip, moe_align_wide_body), bit for bit against the CPU oracle at
the edges of its range, and with the quantisation beside it against shorter calls, which take the single-workgroup form."""
import dataclasses

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("numel,E,bs", [(1024, 128, 16), (1025, 128, 16), (1025, 1, 1), (1087, 271, 160), (1088, 272, 160), (2048, 5, 128),
                                        (2049, 256, 64), (4096, 767, 32), (4096, 768, 32), (16385, 33, 7), (32769, 512, 128),
                                        (65535, 256, 16), (65536, 3, 64), (65537, 128, 64)])
@pytest.mark.parametrize("form", ["plain", "map", "ignore", "local"])
def test_align(oracle, numel, E, bs, form):
    from lightop_amd import op

    dev = torch.device("cuda:0")
    print(f"[case] wide alignment numel={numel} E={E} bs={bs} {form}", flush=True)
    g = torch.Generator().manual_seed(numel + E)
    ids = torch.randint(0, E, (numel, 1), generator=g, dtype=torch.int64)
    ids[: numel // 3] = E // 2                       # one expert with many slots in the first chunks
    ids[[0, numel // 2, numel - 1]] = torch.tensor([[-1], [E], [E - 1]])  # ids that are no expert: slots of none
    emap = None
    if form in ("map", "ignore"):
        emap = torch.where(torch.arange(E) % 3 == 0, torch.arange(E) // 3, -1).to(torch.int32)
    # (the oracle refuses such ids: there they are those of one more expert, which comes last and is on another rank)
    rids = torch.where((ids >= 0) & (ids < E), ids, E).to(torch.int32)
    rmap = torch.cat([torch.arange(E, dtype=torch.int32) if emap is None else emap, torch.tensor([-1], dtype=torch.int32)])
    cap, nb = oracle.align_buffer_sizes(numel, E, bs)
    cap, nb = cap + 77, nb + 3                       # what lies past the last block is padding, too
    for n in ([0, 1, numel // 2, numel] if form == "local" else [None]):
        s = torch.full((cap,), -7, dtype=torch.int32, device=dev)
        e = torch.full((nb,), -7, dtype=torch.int32, device=dev)
        p = torch.full((1,), -7, dtype=torch.int32, device=dev)
        mask = torch.full((numel,), True, dtype=torch.bool, device=dev)
        nlt = None if n is None else torch.tensor([n], dtype=torch.int32, device=dev)
        op.moe_align_block_size(ids.to(torch.int32 if E % 2 else torch.int64).to(dev), E, bs, s, e, p,
                                None if emap is None else emap.to(dev), mask, nlt, form == "ignore")
        torch.cuda.synchronize()
        rs, re, rp = oracle.moe_align_block_size(rids, bs, E + 1, expert_map=rmap, ignore_invalid_experts=form == "ignore",
                                                 **({} if n is None else dict(num_local_tokens=n)))
        last = int((rids[: numel if n is None else n] == E).sum())
        P = rp.item() - (0 if form == "ignore" else (last + bs - 1) // bs * bs)
        assert p.item() == P
        assert torch.equal(s.cpu()[:P], rs[:P]) and bool((s.cpu()[P:] == numel).all())
        assert torch.equal(e.cpu()[: P // bs], re[: P // bs]) and bool((e.cpu()[P // bs:] == -1).all())
        if form != "ignore":
            rank = ids.view(-1).clamp(0, E - 1)
            want = (ids.view(-1) >= 0) & (ids.view(-1) < E) & ((emap[rank] >= 0) if emap is not None else True)
            if n is not None:
                want &= torch.arange(numel) < n
            assert torch.equal(mask.cpu(), want)


@pytest.mark.parametrize("M", [513, 1100, 14336, 14337, 16384, 16385])
@pytest.mark.parametrize("channel,share,dtype", [(False, False, torch.bfloat16), (False, True, torch.float16), (True, True, torch.bfloat16)])
def test_quantisation_beside_it(M, channel, share, dtype):
    """Two slots a token: up to 32768 slots (28672 with quantisation by row) by several workgroups, past that by two launches."""
    from lightop_amd import workloads as wl
    from lightop_amd.moe import fused_experts_impl_int8, get_moe_cache, preshuffle_moe_weight

    dev = torch.device("cuda:0")
    print(f"[case] wide alignment in the whole path M={M} channel={channel} share={share} {dtype}", flush=True)
    layer = dataclasses.replace(wl.TINY, E_global=24 if share else 8, quant="channel" if channel else "block")
    w1, w2, w1s, w2s = wl.make_weights(layer, seed=3, device=dev, gen_device="cuda")
    w1, w2 = preshuffle_moe_weight(w1), preshuffle_moe_weight(w2)
    g = torch.Generator(device=dev).manual_seed(M)
    x = torch.randn((M, layer.H), generator=g, device=dev).to(dtype)
    tw, ids = wl.route(layer, torch.randn((M, layer.E_global), generator=g, device=dev))

    def run(rows):
        return fused_experts_impl_int8(
            x[rows], w1, w2, tw[rows], ids[rows], get_moe_cache(2, 2 * layer.I, layer.H, dev, dtype), use_int8_w8a8=True,
            per_channel_quant=channel, global_num_experts=layer.E_global, expert_map=wl.expert_map_for(layer, dev), w1_scale=w1s,
            w2_scale=w2s, block_shape=None if channel else [128, 128])

    want = torch.cat([run(slice(a, min(a + 512, M))) for a in range(0, M, 512)])
    got = run(slice(0, M))
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("M", [12288, 12289, 12800, 16384])
@pytest.mark.parametrize("channel,ids64,offset", [(False, False, 0), (False, True, 0), (False, False, 1), (True, True, 1)])
def test_long_rows(M, channel, ids64, offset):
    """768 values a slot: past 24576 slots by workgroups of 256 (four ids a load where their address allows it)."""
    from lightop_amd import workloads as wl
    from lightop_amd.moe import fused_experts_impl_int8, get_moe_cache, preshuffle_moe_weight

    dev = torch.device("cuda:0")
    print(f"[case] narrow alignment in the whole path M={M} channel={channel} ids64={ids64} offset={offset}", flush=True)
    layer = dataclasses.replace(wl.TINY, H=1536, I=128, E_global=24, quant="channel" if channel else "block")
    w1, w2, w1s, w2s = wl.make_weights(layer, seed=3, device=dev, gen_device="cuda")
    w1, w2 = preshuffle_moe_weight(w1), preshuffle_moe_weight(w2)
    g = torch.Generator(device=dev).manual_seed(M)
    x = torch.randn((M, layer.H), generator=g, device=dev).to(torch.bfloat16)
    tw, ids = wl.route(layer, torch.randn((M + offset, layer.E_global), generator=g, device=dev))
    ids = (ids.long() if ids64 else ids)[offset:]  # (two ids: half a 16-byte piece)
    tw = tw[offset:]

    def run(rows):
        return fused_experts_impl_int8(
            x[rows], w1, w2, tw[rows], ids[rows], get_moe_cache(2, 2 * layer.I, layer.H, dev, torch.bfloat16), use_int8_w8a8=True,
            per_channel_quant=channel, global_num_experts=layer.E_global, expert_map=wl.expert_map_for(layer, dev), w1_scale=w1s,
            w2_scale=w2s, block_shape=None if channel else [128, 128])

    got = run(slice(0, M))
    some = [slice(a, min(a + 512, M)) for a in sorted({0, M // 3 // 512 * 512, M // 2 // 512 * 512, (M - 1) // 512 * 512})]
    for rows in some:
        assert torch.equal(got[rows].view(torch.int16), run(rows).view(torch.int16))
