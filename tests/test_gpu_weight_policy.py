"""Kernels that choose the cache policy of their weight copies by token block (a block that reads its weights alone, or one of
several of an expert), bit for bit against the CPU oracle: experts of none, few, half a block, a whole one and several blocks of
tokens next to each other, by a low and by a high average of slots per expert."""
import pytest
import torch

from test_gpu_parity import gemm_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs", [64, 128])
@pytest.mark.parametrize("counts", [[1, 64, 0, 65, 128, 0, 0, 129, 48, 300, 2], [300, 300, 16]], ids=["low average", "high average"])
@pytest.mark.parametrize("K", [128, 640])
def test_blocks(oracle, bs, counts, K):
    from lightop_amd.moe import (invoke_fused_moe_gemm1_silu_quant, invoke_fused_moe_kernel_int8, moe_align_block_size,
                                 preshuffle_moe_weight)

    dev = torch.device("cuda:0")
    print(f"[case] block {bs}, {counts}, K={K}", flush=True)
    counts = counts + [0] * 13 if len(counts) > 3 else counts
    E, N, M = len(counts), 256, sum(counts)
    Aq, As, W, Ws, _, tw, _ = gemm_case(bs + K, M, 1, E, E, N, K)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(M, generator=torch.Generator().manual_seed(K))]
    ids = ids.to(torch.int32).view(M, 1)
    rs, re, rp = oracle.moe_align_block_size(ids, bs, E)
    s, e, p = moe_align_block_size(ids.to(dev), bs, E)
    ref = oracle.moe_gemm_block_int8(Aq, As, W, Ws, rs, re, rp, tw, True, 1, M, bs)
    Wd = preshuffle_moe_weight(W.to(dev))
    C = torch.full((M, 1, N), 7.0, dtype=torch.bfloat16, device=dev)
    invoke_fused_moe_kernel_int8(Aq.to(dev), Wd, C, As.to(dev), Ws.to(dev), tw.to(dev), s, e, p, True, 1, {"BLOCK_SIZE_M": bs})
    torch.cuda.synchronize()
    assert torch.equal(C.view(M, N).cpu().view(torch.int16), ref.view(torch.int16))
    c1 = oracle.moe_gemm_block_int8(Aq, As, W, Ws, rs, re, rp, tw, False, 1, M, bs)
    rq, rsc = oracle.per_token_group_quant_int8(oracle.silu_and_mul(c1))
    q, sc = invoke_fused_moe_gemm1_silu_quant(Aq.to(dev), Wd, As.to(dev), Ws.to(dev), tw.to(dev), s, e, p, False, 1, M,
                                              {"BLOCK_SIZE_M": bs})
    torch.cuda.synchronize()
    assert torch.equal(sc.cpu(), rsc) and torch.equal(q.cpu(), rq)
