"""Group quantisation with other floors than the default (`eps`): none, one below and above the values, infinity; bit for bit the
oracle's, which divides."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(x, eps):
    from lightop_amd.quant import per_token_group_quant_int8
    from oracle import cpu_oracle as oracle

    rq, rs = oracle.per_token_group_quant_int8(x, eps=eps)
    q, s = per_token_group_quant_int8(x.cuda(), 128, eps=eps)
    torch.cuda.synchronize()
    assert torch.equal(s.cpu().view(torch.int32), rs.view(torch.int32))
    # (a quotient that is not a number has no integer: the kernels clamp it to -128, the oracle's C cast gives 0)
    with np.errstate(invalid="ignore", divide="ignore"):
        nan = np.isnan(x.float().numpy().reshape(-1, 128) / rs.numpy().reshape(-1, 1)).reshape(x.shape)
    bad = (q.cpu().numpy() != np.where(nan, -128, rq.numpy())).nonzero()
    assert bad[0].size == 0, (bad[0][:5], bad[1][:5])


@pytest.mark.parametrize("eps", [0.0, 1e-12, 1e-10])
def test_small_rows_in_fp32(eps):
    """Maxima down to the smallest denormal: past 2^-126 the reciprocal of their scale is no number."""
    g = torch.Generator().manual_seed(1)
    x = torch.randn(64, 128, generator=g) * 2.0 ** -torch.linspace(20, 149, 64)[:, None]
    print(f"[case] group quantisation of small fp32 rows eps={eps}", flush=True)
    _check(x, eps)
