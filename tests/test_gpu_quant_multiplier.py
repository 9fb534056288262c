"""Group quantisation by one multiplication a value, at the values where a quotient sits on an integer: bit for bit the
oracle's, which divides."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(dtype):
    """Groups of 128 values below (and at) maxima of every mantissa; ends of the range, zeros, infinities, NaN, maxima
    below the floor."""
    step = 1 if dtype == torch.bfloat16 else 8  # 128 mantissas of 2048
    one, full = (0x3F80, 128) if dtype == torch.bfloat16 else (0x3C00, 1024)
    top = torch.arange(one, one + full, step // 8 or 1, dtype=torch.int16).view(dtype).float()
    num = torch.arange(1, 128, dtype=torch.float32)
    near = (top[:, None] * num / 127).to(dtype)                 # the values nearest to an integer quotient
    rows = torch.cat([torch.cat([top[:, None].to(dtype), near], 1),
                      torch.cat([top[:, None].to(dtype), (top[:, None] * (1 - torch.arange(127) / 256)).to(dtype)], 1)])
    signs = torch.where(torch.arange(128) % 3 == 0, -1.0, 1.0)
    rows = (rows.float() * signs).to(dtype)
    scaled = [rows]
    for e in ((-100, -33, 20, 120) if dtype == torch.bfloat16 else (-24, -14, -8, 14)):
        scaled.append((rows.float() * 2.0 ** e).to(dtype))
    odd = torch.zeros(8, 128, dtype=dtype)
    odd[1, 5] = float("inf")
    odd[2, 5], odd[2, 6] = float("nan"), 3.0
    odd[3, 5] = float("-inf")
    odd[4] = torch.finfo(dtype).max
    odd[5] = torch.finfo(dtype).tiny
    odd[6, 7] = torch.tensor(1, dtype=torch.int16).view(dtype)  # the smallest denormal
    odd[7] = 1e-10
    return torch.cat(scaled + [odd])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_group_quant_at_integer_quotients(dtype):
    from lightop_amd.quant import per_token_group_quant_int8
    from oracle import cpu_oracle as oracle

    x = _rows(dtype)
    print(f"[case] group quantisation {dtype} {tuple(x.shape)}", flush=True)
    rq, rs = oracle.per_token_group_quant_int8(x)
    q, s = per_token_group_quant_int8(x.cuda(), 128)
    torch.cuda.synchronize()
    assert np.array_equal(s.cpu().numpy().view(np.int32).ravel(), np.asarray(rs).view(np.int32).ravel())
    # (a quotient that is not a number has no integer: the kernels clamp it to -128, the oracle's C cast gives 0)
    with np.errstate(invalid="ignore"):
        nan = np.isnan(x.float().numpy() / np.asarray(rs).reshape(-1, 1))
    bad = (q.cpu().numpy() != np.where(nan, -128, np.asarray(rq))).nonzero()
    assert bad[0].size == 0, (bad[0][:5], bad[1][:5])
