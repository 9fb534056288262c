"""The quantisation that rides in the alignment's launch against the stages of their own, bit for bit: per row and per group,
both 16-bit types, one and several workgroups for the alignment, rows longer than a workgroup keeps in registers, row counts
that leave part of a workgroup idle."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("per_row", [True, False])
@pytest.mark.parametrize("M,k,E,H", [(1, 2, 4, 128), (5, 8, 8, 8320), (67, 4, 16, 2048), (130, 8, 900, 256), (130, 2, 1600, 384),
                                     (1025, 8, 16, 2176), (4099, 2, 4, 128)])
def test_rides_along(M, k, E, H, per_row, dtype):
    from lightop_amd.moe import (fused_experts_impl_int8, fused_experts_workspace_bytes, fused_experts_workspace_views,
                                 moe_align_block_size)
    from lightop_amd.quant import per_token_group_quant_int8, per_token_quant_int8

    dev, I = torch.device("cuda:0"), 128
    print(f"[case] quant with alignment M={M} k={k} E={E} H={H} rows={per_row} {dtype}", flush=True)
    g = torch.Generator(device=dev).manual_seed(M + H)
    x = torch.randn(M, H, generator=g, device=dev).to(dtype)
    x[M // 3] = 0
    ids = torch.randint(0, E, (M, k), generator=g, device=dev, dtype=torch.int32)
    tw = torch.rand(M, k, generator=g, device=dev)
    w1 = torch.randint(-127, 128, (E, 2 * I, H), generator=g, device=dev, dtype=torch.int8)
    w2 = torch.randint(-127, 128, (E, H, I), generator=g, device=dev, dtype=torch.int8)
    shapes = ((E, 2 * I, 1), (E, H, 1)) if per_row else ((E, 2 * I // 128, H // 128), (E, H // 128, I // 128))
    w1s, w2s = (torch.rand(s, generator=g, device=dev) * 1e-3 + 1e-4 for s in shapes)
    cache13 = torch.empty(M * k * max(2 * I, H), dtype=dtype, device=dev)
    ws = torch.zeros(fused_experts_workspace_bytes(M, k, H, I, E) + 256, dtype=torch.uint8, device=dev)
    fused_experts_impl_int8(x, w1, w2, tw, ids, cache13, use_int8_w8a8=True, per_channel_quant=per_row, w1_scale=w1s,
                            w2_scale=w2s, block_shape=None if per_row else [128, 128], lightop_amd_workspace=ws,
                            lightop_amd_block_size_m=16)
    q, s = per_token_quant_int8(x) if per_row else per_token_group_quant_int8(x, 128)
    srt, eids, ntpp = moe_align_block_size(ids, 16, E)
    torch.cuda.synchronize()
    got = fused_experts_workspace_views(ws, M, k, H, I, E, 16)
    assert torch.equal(got["a1q"], q) and torch.equal(got["a1s"].view(-1)[:s.numel()], s.view(-1))
    assert torch.equal(got["num_tokens_post_pad"], ntpp)
    n = int(ntpp)
    assert torch.equal(got["sorted_ids"][:n], srt[:n]) and torch.equal(got["expert_ids"][:n // 16], eids[:n // 16])
