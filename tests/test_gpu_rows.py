"""The kernel for row-major weights at the edges of its tiles, bit for bit against the CPU oracle: token blocks with one
token, one short of full, full and one over, one and several K blocks, a last weight tile of 64 rows."""
import pytest
import torch

from test_gpu_parity import gemm_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs", [16, 32, 64, 128])
@pytest.mark.parametrize("fill", [1, -1, 0, 1 << 10])
@pytest.mark.parametrize("K", [128, 384, 1024])
def test_row_major_blocks(oracle, bs, fill, K):
    from lightop_amd.gemmopt import moe_gemm_w8a8
    from lightop_amd.moe import (invoke_fused_moe_gemm1_silu_quant, invoke_fused_moe_kernel_int8, moe_align_block_size)

    dev = torch.device("cuda:0")
    count = 1 if fill == 1 else bs + (fill if fill < 0 else 1 if fill > 1 else 0)
    print(f"[case] row-major bs={bs} tokens on expert 0: {count} K={K}", flush=True)
    E, I, M = 2, 128, count + 3
    N = 320 if K != 384 else 2 * I
    Aq, As, W, Ws, _, tw, _ = gemm_case(count + K, M, 1, E, E, N, K)
    Ws = Ws * 30
    ids = torch.ones(M, 1, dtype=torch.int32)
    ids[torch.randperm(M, generator=torch.Generator().manual_seed(count))[:count]] = 0
    rs, re, rp = oracle.moe_align_block_size(ids, bs, E)
    s, e, p = moe_align_block_size(ids.to(dev), bs, E)
    cfg = {"BLOCK_SIZE_M": bs}
    C = torch.full((M, 1, N), 7.0, dtype=torch.bfloat16, device=dev)
    invoke_fused_moe_kernel_int8(Aq.to(dev), W.to(dev), C, As.to(dev), Ws.to(dev), tw.to(dev), s, e, p, True, 1, cfg)
    ref = oracle.moe_gemm_block_int8(Aq, As, W, Ws, rs, re, rp, tw, True, 1, M, bs)
    torch.cuda.synchronize()
    assert torch.equal(C.view(M, -1).cpu().view(torch.int16), ref.view(torch.int16))
    if N == 2 * I:
        c1 = oracle.moe_gemm_block_int8(Aq, As, W, Ws, rs, re, rp, tw, False, 1, M, bs)
        rq, rsc = oracle.per_token_group_quant_int8(oracle.silu_and_mul(c1))
        q, sc = invoke_fused_moe_gemm1_silu_quant(Aq.to(dev), W.to(dev), As.to(dev), Ws.to(dev), tw.to(dev), s, e, p,
                                                  False, 1, M, cfg)
        torch.cuda.synchronize()
        assert torch.equal(sc.cpu(), rsc) and torch.equal(q.cpu(), rq)
    a1, w1 = As[:, :1].contiguous(), torch.rand(E, N, 1) * 1e-2 + 1e-3
    C.fill_(7.0)
    moe_gemm_w8a8(Aq.to(dev), W.to(dev), C, a1.to(dev), w1.to(dev), tw.to(dev), s, e, p, 1, cfg)
    ref = oracle.moe_gemm_w8a8(Aq, a1, W, w1, rs, re, rp, tw, True, 1, M, bs)
    torch.cuda.synchronize()
    assert torch.equal(C.view(M, -1).cpu().view(torch.int16), ref.view(torch.int16))
