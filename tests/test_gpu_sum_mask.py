"""The reduction where a workgroup takes several tokens one after the other and asks for the next one's mask ahead, bit for bit
against the CPU oracle: every unrolled slot count and the general one, a last column block that is not full, padded batches."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 2, 3, 4, 6, 8])
@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("local", [None, 0, 1, 1399])
def test_masked(oracle, k, with_bias, local):
    from lightop_amd.moe import moe_sum

    dev = torch.device("cuda:0")
    M, H = 1400, 12296  # seven blocks of 2048 columns, 585 tokens at a time
    print(f"[case] masked sum k={k} bias={with_bias} local={local}", flush=True)
    g = torch.Generator().manual_seed(k)
    x = torch.randn(M, k, H, generator=g, dtype=torch.float32).to(torch.bfloat16)
    b = torch.randn(M, H, generator=g).to(torch.bfloat16) if with_bias else None
    mask = torch.rand(M, k, generator=g) > 0.7
    prev = torch.full((M, H), 3.0, dtype=torch.bfloat16)
    kept = torch.where(mask[..., None], x, torch.zeros_like(x))
    ref = oracle.moe_sum(kept, b, 2.5) if local is None else oracle.moe_sum(kept, b, 2.5, num_local_tokens=local, out=prev)
    out = prev.clone().to(dev)
    x[~mask] = float("nan")
    moe_sum(x.to(dev), out, None if b is None else b.to(dev), expert_mask=mask.reshape(-1).to(dev), factor=2.5,
            num_local_tokens=None if local is None else torch.tensor([local], dtype=torch.int32, device=dev))
    torch.cuda.synchronize()
    assert torch.equal(out.cpu().view(torch.int16), ref.view(torch.int16))
