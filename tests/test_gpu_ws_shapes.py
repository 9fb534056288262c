"""The weight-streaming kernel at the edges of its workgroup shapes, bit for bit against the CPU oracle: two and four
fragments per wave (outputs up to and past 4096), a last tile that is not full, two and four K blocks in flight (K up to and
past 4096) with K blocks that do not fill the ring."""
import pytest
import torch

from test_gpu_parity import gemm_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [112, 4096, 4112])
@pytest.mark.parametrize("K", [128, 384])
@pytest.mark.parametrize("bs", [16, 32])
def test_plain(oracle, bs, K, N):
    from lightop_amd.moe import invoke_fused_moe_kernel_int8, moe_align_block_size, preshuffle_moe_weight

    dev = torch.device("cuda:0")
    print(f"[case] weight streaming plain bs={bs} K={K} N={N}", flush=True)
    M, E = bs + 4, 2
    Aq, As, W, Ws, _, tw, _ = gemm_case(N + K, M, 1, E, E, N, K)
    ids = torch.ones(M, 1, dtype=torch.int32)
    ids[:3] = 0
    rs, re, rp = oracle.moe_align_block_size(ids, bs, E)
    s, e, p = moe_align_block_size(ids.to(dev), bs, E)
    C = torch.full((M, 1, N), 7.0, dtype=torch.bfloat16, device=dev)
    invoke_fused_moe_kernel_int8(Aq.to(dev), preshuffle_moe_weight(W.to(dev)), C, As.to(dev), Ws.to(dev), tw.to(dev), s, e, p,
                                 True, 1, {"BLOCK_SIZE_M": bs})
    ref = oracle.moe_gemm_block_int8(Aq, As, W, Ws, rs, re, rp, tw, True, 1, M, bs)
    torch.cuda.synchronize()
    assert torch.equal(C.view(M, -1).cpu().view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("K", [128, 640, 4096, 4224])
@pytest.mark.parametrize("bs", [16, 32])
def test_fused(oracle, bs, K):
    from lightop_amd.moe import invoke_fused_moe_gemm1_silu_quant, moe_align_block_size, preshuffle_moe_weight

    dev = torch.device("cuda:0")
    print(f"[case] weight streaming fused bs={bs} K={K}", flush=True)
    M, E, N = bs + 4, 2, 256
    Aq, As, W, Ws, _, tw, _ = gemm_case(K, M, 1, E, E, N, K)
    Ws = Ws * 10
    ids = torch.ones(M, 1, dtype=torch.int32)
    ids[:3] = 0
    rs, re, rp = oracle.moe_align_block_size(ids, bs, E)
    s, e, p = moe_align_block_size(ids.to(dev), bs, E)
    c1 = oracle.moe_gemm_block_int8(Aq, As, W, Ws, rs, re, rp, tw, False, 1, M, bs)
    rq, rsc = oracle.per_token_group_quant_int8(oracle.silu_and_mul(c1))
    q, sc = invoke_fused_moe_gemm1_silu_quant(Aq.to(dev), preshuffle_moe_weight(W.to(dev)), As.to(dev), Ws.to(dev), tw.to(dev),
                                              s, e, p, False, 1, M, {"BLOCK_SIZE_M": bs})
    torch.cuda.synchronize()
    assert torch.equal(sc.cpu(), rsc) and torch.equal(q.cpu(), rq)
