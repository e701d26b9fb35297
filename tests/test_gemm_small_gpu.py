"""The GEMM's small output tiles: few rows or columns, and the last rows of a tall
product.  Each K sum runs in the same order as on 256 x 256 tiles, so the results are
held to those bit for bit; at sizes that only run on small tiles, to the float64
product of the dequantised operands."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

F8 = torch.float8_e4m3fn


def _lib():
    from sr_dit import _lib
    return _lib


def _operands(M, N, K, rs, seed):
    g = torch.Generator("cpu").manual_seed(seed)
    a = (torch.randn(M, K, generator=g) * 0.6).to(F8).cuda()
    b = (torch.randn(N, K, generator=g) * 0.6).to(F8).cuda()
    sa = (torch.rand(M if rs else 1, generator=g) + 0.5).cuda()
    sb = (torch.rand(N if rs else 1, generator=g) / 64 + 1 / 128).cuda()
    bias = (torch.randn(N, generator=g) * 2).to(torch.bfloat16).cuda()
    return a, b, sa, sb, bias


@pytest.mark.parametrize("rs", [False, True], ids=["tensor", "rowwise"])
@pytest.mark.parametrize("M,N,K", [(1, 16, 128), (64, 64, 256), (65, 80, 384), (33, 1040, 512),
                                   (129, 48, 3072), (640, 3072, 128), (700, 6160, 256)])
def test_small_tiles_match_the_dequantised_product(M, N, K, rs):
    """Per element within half a bf16 ulp (2^-8 relative) and the fp32 sum's 2^-12 of
    the sum of |terms|; the padding of a strided output is left alone."""
    print(f"[case] small gemm M={M} N={N} K={K} rowwise={rs}", flush=True)
    a, b, sa, sb, bias = _operands(M, N, K, rs, M + N + K)
    buf = torch.full((M, N + 16), 7.0, dtype=torch.bfloat16, device="cuda")
    _lib().fp8_gemm(a, b, sa, sb, bias, buf[:, :N])
    torch.cuda.synchronize()
    scale = sa.double().reshape(-1, 1) * sb.double().reshape(1, -1)
    ref = torch.matmul(a.double(), b.double().T.contiguous()) * scale + bias.double()
    terms = torch.matmul(a.double().abs(), b.double().abs().T.contiguous()) * scale
    err = (buf[:, :N].double() - ref).abs()
    assert (err <= 2.0 ** -8 * ref.abs() + 2.0 ** -12 * (terms + bias.double().abs())).all()
    assert (buf[:, N:] == 7.0).all()


@pytest.mark.parametrize("M,pad,K,epilogue", [
    (1, 8192, 1024, 0), (257, 8192, 384, 1), (512, 8192, 3072, 2), (2048, 8192, 256, 0),
    # 22 tile rows of 12: the last row of tiles opens a second round of 256 CUs
    (5424, 5632, 1024, 1), (5377, 5632, 1024, 2), (5631, 5632, 1152, 0)])
def test_small_tiles_equal_large_tiles(M, pad, K, epilogue):
    """The first M rows of a product that runs on 256 x 256 tiles alone (``pad`` rows),
    with per-row scales; epilogue 1 GELU and the amax, 2 the largest positive value."""
    print(f"[case] small against large tiles M={M} K={K} epilogue={epilogue}", flush=True)
    L, N = _lib(), 3072
    a, b, sa, sb, bias = _operands(pad, N, K, True, M + K)
    ep = {0: 0, 1: 1, 2: L.GEMM_AMAX_POS}[epilogue]
    outs, words = [], []
    for rows in (M, pad):
        out = torch.full((rows, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        word = torch.full((1,), 12345, dtype=torch.int32, device="cuda") if epilogue else None
        L.fp8_gemm_ex(a[:rows], b, sa[:rows], sb, bias, out, epilogue=ep, amax_out=word,
                      split_tail=False)
        outs.append(out)
        words.append(word)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1][:M])
    if epilogue == 1:
        assert words[0].view(torch.float32).item() == outs[0].float().abs().max().item()
    elif epilogue == 2:
        assert words[0].view(torch.float32).item() == outs[0].float().max().item()


def test_small_tiles_split_output():
    """Column blocks in tensors of their own, on small tiles and in the remainder rows."""
    print("[case] small gemm split output", flush=True)
    L = _lib()
    for M, G, W, K in ((100, 3, 256, 256), (5424, 2, 1536, 1024)):
        a, b, sa, sb, bias = _operands(M, G * W, K, True, M)
        out = torch.full((G, M, W), float("nan"), dtype=torch.bfloat16, device="cuda")
        want = torch.empty(M, G * W, dtype=torch.bfloat16, device="cuda")
        L.fp8_gemm_split(a, b, sa, sb, bias, out)
        L.fp8_gemm(a, b, sa, sb, bias, want)
        torch.cuda.synchronize()
        assert torch.equal(out.permute(1, 0, 2).reshape(M, G * W), want), M


@pytest.mark.parametrize("M,N,K,gelu", [(1, 16, 64, False), (512, 3072, 4096, True),
                                        (65, 1536, 192, False), (1000, 3072, 128, True),
                                        (2500, 3072, 512, False),
                                        # two K groups: 24 and 26 stages, 64- and 128-row
                                        # tiles, ragged rows and columns; 25 stages: one
                                        (1, 16, 1536, False), (130, 1040, 1664, True),
                                        (500, 3056, 1536, True), (385, 3072, 1600, False)])
def test_bf16_small_tiles_match_float64(M, N, K, gelu):
    """bf16 operands: the fp32 sum's K 2^-24 of the sum of |terms|, half an ulp of the
    rounding, and a full one where the GELU reads a value at a rounding boundary."""
    print(f"[case] bf16 small M={M} N={N} K={K} gelu={gelu}", flush=True)
    g = torch.Generator("cpu").manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
    bias = (torch.randn(N, generator=g) * 0.3).to(torch.bfloat16).cuda()
    out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    _lib().bf16_linear(a, w, bias, out, gelu=gelu)
    torch.cuda.synchronize()
    ref = torch.matmul(a.double(), w.double().T.contiguous()) + bias.double()
    terms = torch.matmul(a.double().abs(), w.double().abs().T.contiguous()) + bias.double().abs()
    slack = (K + 1) * 2.0 ** -24 * terms + 2.0 ** -8 * ref.abs()
    if gelu:  # |GELU'| <= 1.13; its own rounding is another half ulp
        ref = torch.nn.functional.gelu(ref, approximate="tanh")
        slack = 1.13 * slack + 2.0 ** -8 * ref.abs() + 1e-6
    assert ((out.double() - ref).abs() <= slack + 1e-30).all()
