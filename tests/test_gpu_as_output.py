"""Stores of the activation-stationary GEMM (csrc/gemm_as.hip) through a descriptor of the output: the last rows and the memory
behind them, pieces of padding, fp16, slots of another rank's expert, and an output that a descriptor does not address."""
import pytest
import torch

from test_gpu_fold_scales import oracle_rows
from test_gpu_parity import gemm_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs,K,N,dtype", [(64, 768, 64, torch.bfloat16), (128, 768, 832, torch.float16), (128, 512, 320, torch.float16),
                                          (64, 768, 26624, torch.bfloat16), (128, 768, 33216, torch.bfloat16)])  # 3.5e9, 4.4e9 bytes
def test_rows_and_extent(oracle, bs, K, N, dtype):
    from lightop_amd.moe import invoke_fused_moe_kernel_int8, moe_align_block_size, preshuffle_moe_weight

    dev = torch.device("cuda:0")
    print(f"[case] activation-stationary output bs={bs} K={K} N={N} {dtype}", flush=True)
    M, E = 66001, 2  # (the shortest launch that takes this kernel)
    Aq, As, W, Ws, _, tw, _ = gemm_case(N + bs, M, 1, E, E, N, K)
    ids = (torch.arange(M) % 5 == 0).to(torch.int32).view(M, 1)
    emap = None
    if N == 832:  # every tenth token's expert is on another rank: rows of zeros
        ids[::10] = 2
        emap = torch.tensor([0, 1, -1], dtype=torch.int32)
    rows = torch.cat([torch.arange(40), torch.arange(40, M - 70, 4093), torch.arange(M - 70, M)])
    local = ids[rows].view(-1) < 2
    ref = oracle_rows(oracle, Aq, As, W, Ws, tw, ids.clamp(max=1), rows)
    s, e, p = moe_align_block_size(ids.to(dev), bs, 3 if emap is not None else E,
                                   **({} if emap is None else {"expert_map": emap.to(dev)}))
    buf = torch.full((M + 4, 1, N), 7.0, dtype=dtype, device=dev)
    invoke_fused_moe_kernel_int8(Aq.to(dev), preshuffle_moe_weight(W.to(dev)), buf[:M], As.to(dev), Ws.to(dev), tw.to(dev), s, e, p,
                                 True, 1, {"BLOCK_SIZE_M": bs})
    torch.cuda.synchronize()
    got = buf.view(M + 4, N)[torch.cat([rows, torch.arange(M, M + 4)]).to(dev)].cpu()
    assert bool((got[len(rows):] == 7.0).all())
    got = got[: len(rows)]
    assert bool((got[~local] == 0).all())
    want = ref[local]
    if dtype == torch.float16:  # the oracle's rows are bf16 of the same fp32 sums: half an ulp of that
        assert bool(((got[local].float() - want.float()).abs() <= want.float().abs() * 2.0 ** -8 + 2.0 ** -24).all())
    else:
        assert torch.equal(got[local].view(torch.int16), want.view(torch.int16))
