"""The head's fp32 Linear on bf16 MFMAs (its input cut into three exact pieces) against
float64, at the edges of its tiles and with values that need all three pieces, and its
non-finite inputs against the fp32 product's."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

U32 = 2.0 ** -24


def _lib():
    from sr_dit import _lib
    return _lib


def _inputs(M, N, K, mod_dtype, spread, seed):
    g = torch.Generator("cpu").manual_seed(seed)
    a = (torch.randn(M, K, generator=g) * torch.exp(spread * torch.randn(M, 1, generator=g)))
    a = a.to(torch.bfloat16).cuda()
    mod = (torch.randn(1, 2, K, generator=g) * 0.3).to(mod_dtype).cuda()
    e = (torch.randn(1, K, generator=g) * 0.3).cuda()
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
    b = torch.randn(N, generator=g).to(torch.bfloat16).cuda()
    return a, mod, e, w, b


def _vectors(mod, e):
    m = mod.float() + e.unsqueeze(1)
    return (1 + m[0, 1]).contiguous(), m[0, 0].contiguous()


@pytest.mark.parametrize("M,N,K,pad", [(1, 1, 64, 0), (63, 64, 128, 0), (65, 66, 192, 2),
                                       (200, 192, 3072, 0), (2600, 200, 256, 0), (17, 37, 4096, 3)])
@pytest.mark.parametrize("mod_dtype,spread", [(torch.bfloat16, 0.0), (torch.float32, 6.0)],
                         ids=["bf16", "fp32-wide"])
def test_head_linear_matches_float64(M, N, K, pad, mod_dtype, spread):
    """xin rounds twice in fp32 as torch's kernels round it; then K fp32 additions and
    the final one: (K + 2) 2^-24 of the sum of |terms|."""
    print(f"[case] head linear M={M} N={N} K={K} {mod_dtype}", flush=True)
    a, mod, e, w, b = _inputs(M, N, K, mod_dtype, spread, M + N + K)
    buf = torch.full((M, N + pad), 7.0, device="cuda")
    _lib().head_linear(a, mod, e, w, b, buf[:, :N])
    s1, m0 = _vectors(mod, e)
    xin = (a.float() * s1 + m0).double()
    ref = torch.matmul(xin, w.double().T.contiguous()) + b.double()
    terms = torch.matmul(xin.abs(), w.double().abs().T.contiguous()) + b.double().abs()
    torch.cuda.synchronize()
    assert ((buf[:, :N].double() - ref).abs() <= (K + 2) * U32 * terms).all()
    assert (buf[:, N:] == 7.0).all()
    # the entry that is given the vectors forms the same product, in the same order
    # where it takes the same kernel (up to 64 columns, or 2560 rows of 192)
    out = torch.empty(M, N, device="cuda")
    _lib().linear_f32_modulated(a, s1, m0, w, b, out)
    torch.cuda.synchronize()
    assert ((out.double() - ref).abs() <= (K + 2) * U32 * terms).all()
    if N <= 64 or M >= 2560:
        assert torch.equal(out, buf[:, :N])
    # two pieces (16 bits of xin) would miss the bound's typical error by far
    if spread == 0.0 and K >= 256:
        cut = (xin.float().view(torch.int32) & -256).view(torch.float32).double()
        off = (torch.matmul(cut, w.double().T.contiguous()) + b.double() - ref).norm()
        assert (buf[:, :N].double() - ref).norm() < 0.3 * off


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.3e38])
def test_head_linear_non_finite_rows(value):
    """A non-finite or overflowing xin gives the infinity or NaN that the fp32 product
    gives, in its row alone."""
    print(f"[case] head linear {value}", flush=True)
    a, mod, e, w, b = _inputs(70, 64, 128, torch.float32, 0.0, 5)
    mod.zero_(), e.zero_()
    e[0, 3] = 1.0                                   # s1[3] = 2: the large value overflows
    a[66, 3] = value
    out = torch.empty(70, 64, device="cuda")
    _lib().head_linear(a, mod, e, w, b, out)
    s1, m0 = _vectors(mod, e)
    xin = (a.float() * s1 + m0)
    ref = torch.matmul(xin.cpu(), w.float().cpu().T.contiguous()) + b.float().cpu()
    got = out.cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    assert torch.equal(torch.isinf(got), torch.isinf(ref))
    assert torch.equal(got[torch.isinf(ref)], ref[torch.isinf(ref)])
    keep = torch.arange(70) != 66
    assert torch.isfinite(got[keep]).all()
