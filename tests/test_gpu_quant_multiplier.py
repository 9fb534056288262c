"""Group quantisation by one multiplication a value, at the values where a quotient sits on an integer: bit for bit the
oracle's, which divides."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(dtype):
    """Groups of 128 values below (and at) maxima of every mantissa; ends of the range, zeros, infinities, NaN, maxima
    below the floor."""
    one, full = (0x3F80, 128) if dtype == torch.bfloat16 else (0x3C00, 1024)
    top = torch.arange(one, one + full, dtype=torch.int16).view(dtype).float()
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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_activation_and_quantisation_at_integer_quotients(dtype):
    """Behind a gate of 256, whose SiLU is 256: the activation is the other half, scaled."""
    from lightop_amd.moe import act_and_mul_group_quant
    from oracle import cpu_oracle as oracle

    up = _rows(dtype)
    up = up[up.float().abs().amax(1) < 64]  # (what stays finite when it is scaled)
    c1 = torch.cat([torch.full_like(up, 256.0), up], 1)
    print(f"[case] activation and group quantisation {dtype} {tuple(c1.shape)}", flush=True)
    rq, rs = oracle.per_token_group_quant_int8(oracle.silu_and_mul(c1))
    q, s = act_and_mul_group_quant(c1.cuda(), "silu")
    torch.cuda.synchronize()
    ok = torch.isfinite(c1.float()).all(1)
    assert torch.equal(s.cpu()[ok], rs[ok]) and torch.equal(q.cpu()[ok], rq[ok])


@pytest.mark.parametrize("int4,bs", [(False, 16), (False, 32), (False, 64), (False, 128), (False, 160), (True, 16), (True, 32),
                                     (True, 64), (True, 128)])
@pytest.mark.parametrize("special", [False, True])
def test_fused_epilogues_at_integer_quotients(int4, bs, special):
    """Column j of the activation is j / 127 of the row's maximum before its rounding to 16 bits, rows are scaled by every bf16
    mantissa and more.  special: among them rows with infinite and NaN gates and with a maximum other than zero below 1e-10, for
    which the tile (or the lane) divides."""
    from lightop_amd import _lib
    from lightop_amd.moe import (invoke_fused_moe_gemm1_silu_quant, moe_align_block_size, preshuffle_moe_scale_int4,
                                 preshuffle_moe_weight, preshuffle_moe_weight_int4)
    from oracle import cpu_oracle as oracle

    dev = torch.device("cuda:0")
    print(f"[case] fused first stage int4={int4} bs={bs} special={special}", flush=True)
    M, I, K = 700, 128, 128
    Aq = torch.zeros(M, K, dtype=torch.int8)
    Aq[:, 0], Aq[:, 1], Aq[:, 2] = 1, 8, 64
    j = torch.arange(I)
    W = torch.zeros(1, 2 * I, K, dtype=torch.int8)
    W[0, :I, 0], W[0, :I, 1], W[0, :I, 2] = 7, 7, 1  # the gate, 127 times the row's scale
    W[0, I:, 0], W[0, I:, 1], W[0, I:, 2] = (j % 8).to(torch.int8), (j // 8 % 8).to(torch.int8), (j // 64).to(torch.int8)
    scales = 1 + torch.arange(M) / 640
    if special:
        scales[::37] = 2.0 ** -22       # gate 3e-5, activation below 3.5e-10 / 8
        scales[5::150] = float("inf")
        scales[77::150] = float("nan")
    As = scales.reshape(M, 1).contiguous()
    ids, tw = torch.zeros(M, 1, dtype=torch.int32), torch.ones(M, 1)
    rs, re, rp = oracle.moe_align_block_size(ids, bs, 1)
    s, e, p = moe_align_block_size(ids.to(dev), bs, 1)
    if int4:
        W4 = oracle.pack_int4(W)
        Ws = torch.cat([torch.ones(1, I, 1), torch.full((1, I, 1), 1 / 128)], 1)
        c1 = oracle.moe_gemm_w4a8(Aq, As, W4, Ws, rs, re, rp, tw, False, 1, M, bs)
        Wx, Wsx, flags = preshuffle_moe_weight_int4(W4.to(dev)), preshuffle_moe_scale_int4(Ws.to(dev)), _lib.LO_GEMM_W4
    else:
        Ws = torch.tensor([1.0, 1 / 128]).reshape(1, 2, 1)
        c1 = oracle.moe_gemm_block_int8(Aq, As, W, Ws, rs, re, rp, tw, False, 1, M, bs)
        Wx, Wsx, flags = preshuffle_moe_weight(W.to(dev)), Ws.to(dev), 0
    act = oracle.silu_and_mul(c1)
    rq, rsc = oracle.per_token_group_quant_int8(act)
    ok = torch.isfinite(scales)
    peak = act[ok].float().abs().amax(1)
    assert bool((peak < 1e-10).any()) == special and bool((peak > 0).all())
    q, sc = invoke_fused_moe_gemm1_silu_quant(Aq.to(dev), Wx, As.to(dev), Wsx, tw.to(dev), s, e, p, False, 1, M,
                                              {"BLOCK_SIZE_M": bs}, fused_scale=False, flags=flags)
    torch.cuda.synchronize()
    assert torch.equal(sc.cpu()[ok], rsc[ok]) and torch.equal(q.cpu()[ok], rq[ok])
