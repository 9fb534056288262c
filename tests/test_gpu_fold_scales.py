"""The fold without a conversion (csrc/gemm.h, fold_biased) at the ends of the scales it takes, and the conversion it gives way to
past them, bit for bit against the CPU oracle: in every kernel that folds that way, with the extreme scale on one token or
one weight block of one K block, with sums at their extremes, and with scales of either sign and zero."""
import pytest
import torch

from test_gpu_parity import gemm_case

pytestmark = pytest.mark.gpu

BELOW = 1.0 - 2.0 ** -24  # (rounds to the float below one)
# name -> (token scale, weight scale) of the marked entries; None: as drawn
SCALES = {
    "token smallest": (2.0 ** -62, None), "token too small": (2.0 ** -62 * BELOW, None),
    "token largest": (2.0 ** 43 * BELOW, None), "token too large": (2.0 ** 43, None), "token zero": (0.0, None),
    "token negative": (-0.03, None), "token denormal": (2.0 ** -140, None), "token far too large": (2.0 ** 100, 2.0 ** -60),
    "weight largest": (None, 2.0 ** 64 * BELOW), "weight too large": (None, 2.0 ** 64), "weight negative": (None, -0.01),
    "weight denormal": (None, 2.0 ** -140), "weight zero": (None, 0.0), "both ends": (2.0 ** -62, 2.0 ** 64 * BELOW),
}
# tokens on expert 0, block size, form
KERNELS = [(40, 64, "shuffled"), (100, 128, "shuffled"), (128, 128, "shuffled"), (90, 160, "shuffled"), (160, 160, "shuffled"),
           (10, 16, "rows"), (30, 32, "rows"), (60, 64, "rows"), (128, 128, "rows"), (40, 64, "int4"), (100, 128, "int4"),
           (90, 160, "int4"), (160, 160, "int4"), (66000, 64, "shuffled"), (66000, 128, "shuffled")]


@pytest.mark.parametrize("count,bs,form", KERNELS)
@pytest.mark.parametrize("K", [128, 384])
def test_plain(oracle, count, bs, form, K):
    from lightop_amd import _lib
    from lightop_amd.moe import (invoke_fused_moe_kernel_int8, moe_align_block_size, preshuffle_moe_scale_int4,
                                 preshuffle_moe_weight, preshuffle_moe_weight_int4)

    dev = torch.device("cuda:0")
    large = count > 1000  # enough token blocks for the activation-stationary kernel
    E, N, M = 2, 64 if large else 320, count + 5
    names = ["token largest", "token too large", "weight too large", "both ends"] if large else list(SCALES)
    Aq, As, W, Ws, _, tw, _ = gemm_case(count + K, M, 1, E, E, N, K)
    Ws = Ws * 10
    if form == "int4":
        W = torch.randint(0, 256, (E, N, K // 2), generator=torch.Generator().manual_seed(count), dtype=torch.int16).to(torch.uint8)
        Ws = Ws.repeat_interleave(128, dim=1)[:, :N].contiguous()
    Aq[0], Aq[1] = 127, -128  # sums at their extremes
    if form != "int4":
        W[0, 0], W[0, 1] = 127, -128
    ids = torch.zeros(M, 1, dtype=torch.int32)
    ids[torch.arange(2, M - 3, max(1, (M - 5) // 5))[:5]] = 1
    rs, re, rp = oracle.moe_align_block_size(ids, bs, E)
    s, e, p = moe_align_block_size(ids.to(dev), bs, E)
    if form == "int4":
        Wd, flags = preshuffle_moe_weight_int4(W.to(dev)), _lib.LO_GEMM_W4
    else:
        Wd, flags = (preshuffle_moe_weight(W.to(dev)) if form == "shuffled" else W.to(dev)), 0
    for name in names:
        ts, ws = SCALES[name]
        print(f"[case] {form} bs={bs} count={count} K={K} {name}", flush=True)
        A2, W2 = As.clone(), Ws.clone()
        if ts is not None:
            A2[[0, 1, M - 1], K // 128 - 1] = ts
        if ws is not None:
            W2[0, [0, -1], K // 128 - 1] = ws
        if form == "int4":
            ref = oracle.moe_gemm_w4a8(Aq, A2, W, W2, rs, re, rp, tw, True, 1, M, bs)
        else:
            ref = oracle.moe_gemm_block_int8(Aq, A2, W, W2, rs, re, rp, tw, True, 1, M, bs)
        C = torch.full((M, 1, N), 7.0, dtype=torch.bfloat16, device=dev)
        Wsd = preshuffle_moe_scale_int4(W2.to(dev)) if form == "int4" else W2.to(dev)
        invoke_fused_moe_kernel_int8(Aq.to(dev), Wd, C, A2.to(dev), Wsd, tw.to(dev), s, e, p, True, 1, {"BLOCK_SIZE_M": bs}, flags=flags)
        torch.cuda.synchronize()
        got = C.view(M, N).cpu()
        assert bool(ref.float().isfinite().all())
        assert torch.equal(got.view(torch.int16), ref.view(torch.int16)), name


@pytest.mark.parametrize("bs,form", [(64, "shuffled"), (128, "shuffled"), (160, "shuffled"), (128, "rows"), (128, "int4"), (160, "int4")])
@pytest.mark.parametrize("scale", [2.0 ** 60, -2.0 ** 44])
def test_fused(oracle, bs, form, scale):
    """A first stage whose tiles redo their sums before the activation."""
    from lightop_amd import _lib
    from lightop_amd.moe import (invoke_fused_moe_gemm1_silu_quant, moe_align_block_size, preshuffle_moe_scale_int4,
                                 preshuffle_moe_weight, preshuffle_moe_weight_int4)

    dev = torch.device("cuda:0")
    print(f"[case] fused {form} bs={bs} scale={scale}", flush=True)
    M, E, N, K = 2 * bs - 7, 2, 512, 384
    Aq, As, W, Ws, _, tw, _ = gemm_case(bs, M, 1, E, E, N, K)
    Ws = Ws * 10
    if form == "int4":
        W = torch.randint(0, 256, (E, N, K // 2), generator=torch.Generator().manual_seed(bs), dtype=torch.int16).to(torch.uint8)
        Ws = Ws.repeat_interleave(128, dim=1)[:, :N].contiguous()
    As[::3, 1] = scale
    Aq[::3, 128:256] = 0  # (its products are zero: the sums stay where SiLU is neither zero nor the identity)
    ids = (torch.arange(M) % 4 == 0).to(torch.int32).view(M, 1)
    rs, re, rp = oracle.moe_align_block_size(ids, bs, E)
    s, e, p = moe_align_block_size(ids.to(dev), bs, E)
    if form == "int4":
        c1 = oracle.moe_gemm_w4a8(Aq, As, W, Ws, rs, re, rp, tw, False, 1, M, bs)
        Wd, Wsd, flags = preshuffle_moe_weight_int4(W.to(dev)), preshuffle_moe_scale_int4(Ws.to(dev)), _lib.LO_GEMM_W4
    else:
        c1 = oracle.moe_gemm_block_int8(Aq, As, W, Ws, rs, re, rp, tw, False, 1, M, bs)
        Wd, Wsd, flags = preshuffle_moe_weight(W.to(dev)) if form == "shuffled" else W.to(dev), Ws.to(dev), 0
    rq, rsc = oracle.per_token_group_quant_int8(oracle.silu_and_mul(c1))
    q, sc = invoke_fused_moe_gemm1_silu_quant(Aq.to(dev), Wd, As.to(dev), Wsd, tw.to(dev), s, e, p, False, 1, M,
                                              {"BLOCK_SIZE_M": bs}, flags=flags)
    torch.cuda.synchronize()
    assert torch.equal(sc.cpu(), rsc) and torch.equal(q.cpu(), rq)


@pytest.mark.parametrize("name", ["as drawn", "token too large", "weight too large", "both ends"])
@pytest.mark.parametrize("bs,K", [(64, 768), (128, 768), (64, 256), (128, 1024)])
def test_activation_stationary(oracle, bs, K, name):
    """Several weight tiles a workgroup, the last of them 64 rows wide, with the number of K blocks known to the compiler and not."""
    from lightop_amd.moe import invoke_fused_moe_kernel_int8, moe_align_block_size, preshuffle_moe_weight

    dev = torch.device("cuda:0")
    print(f"[case] activation-stationary bs={bs} K={K} {name}", flush=True)
    M, E, N = 66000, 2, 832  # (the shortest launch that takes this kernel)
    Aq, As, W, Ws, _, tw, _ = gemm_case(K + bs, M, 1, E, E, N, K)
    Ws = Ws * 10
    ts, ws = SCALES.get(name, (None, None))
    if ts is not None:
        As[[0, 1, M - 1], K // 128 - 1] = ts
    if ws is not None:
        Ws[0, [0, -1], K // 128 - 1] = ws
    ids = (torch.arange(M) % 5 == 0).to(torch.int32).view(M, 1)
    # checked on some of the tokens, those with a marked scale and their neighbours among them: a row depends on no other
    rows = torch.cat([torch.arange(150), torch.arange(150, M - 150, 1021), torch.arange(M - 150, M)])
    ref = oracle_rows(oracle, Aq, As, W, Ws, tw, ids, rows)
    s, e, p = moe_align_block_size(ids.to(dev), bs, E)
    C = torch.full((M, 1, N), 7.0, dtype=torch.bfloat16, device=dev)
    invoke_fused_moe_kernel_int8(Aq.to(dev), preshuffle_moe_weight(W.to(dev)), C, As.to(dev), Ws.to(dev), tw.to(dev), s, e, p, True, 1,
                                 {"BLOCK_SIZE_M": bs})
    torch.cuda.synchronize()
    got = C.view(M, N).cpu()[rows]
    assert bool(ref.float().isfinite().all())
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))


def oracle_rows(oracle, Aq, As, W, Ws, tw, ids, rows):
    """The rows of a GEMM with one slot a token, computed alone."""
    A, S, w, i = (t[rows].contiguous() for t in (Aq, As, tw, ids))
    s, e, p = oracle.moe_align_block_size(i, 64, W.shape[0])
    return oracle.moe_gemm_block_int8(A, S, W, Ws, s, e, p, w, True, 1, len(rows), 64)
