"""The top-k reduction of rows of more than 4096 values (csrc/elementwise.hip): on either side of the line from which its workgroups
have 512 threads, with a mask (several tokens each) and without (one), bit for bit against the CPU oracle."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,H,k", [(512, 7168, 8), (513, 7168, 8), (1025, 7168, 8), (683, 4104, 2), (1366, 4096, 8), (700, 8200, 3),
                                   (2050, 7168, 1)])
@pytest.mark.parametrize("masked,biased", [(False, False), (True, True), (True, False)])
def test_wide_rows(oracle, M, H, k, masked, biased):
    from lightop_amd import op

    dev = torch.device("cuda:0")
    print(f"[case] moe_sum M={M} H={H} k={k} masked={masked} biased={biased}", flush=True)
    g = torch.Generator().manual_seed(M + H + k)
    x = torch.randn(M, k, H, generator=g).to(torch.bfloat16)
    bias = torch.randn(M, H, generator=g).to(torch.bfloat16) if biased else None
    mask = torch.rand(M, k, generator=g) < 0.4 if masked else None
    for n in (None, M // 2 + 1):
        prev = torch.full((M, H), 3.0, dtype=torch.bfloat16)
        out = prev.clone().to(dev)
        nlt = None if n is None else torch.tensor([n], dtype=torch.int32, device=dev)
        op.moe_sum(x.to(dev), out, None if bias is None else bias.to(dev), None if mask is None else mask.to(dev), nlt, 1.5)
        torch.cuda.synchronize()
        zeroed = x if mask is None else torch.where(mask[..., None], x, torch.zeros((), dtype=x.dtype))
        ref = oracle.moe_sum(zeroed, bias, 1.5, **({} if n is None else dict(num_local_tokens=n, out=prev)))
        assert torch.equal(out.cpu().view(torch.int16), ref.view(torch.int16)), n
