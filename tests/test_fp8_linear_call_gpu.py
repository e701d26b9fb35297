"""Fp8Linear's one call against its quantiser and its GEMM called one after the other."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scaling", ["rowwise", "tensor"])
@pytest.mark.parametrize("shape,dtype,bias", [((1, 128), torch.bfloat16, True),
                                              ((3, 7, 256), torch.float32, False),
                                              ((300, 384), torch.float16, True),
                                              ((5424, 1024), torch.bfloat16, True)])
def test_fp8_linear_equals_quantiser_and_gemm(scaling, shape, dtype, bias):
    from sr_dit import _lib
    from sr_dit import fp8_linear as fl
    print(f"[case] fp8 linear call {shape} {dtype} {scaling}", flush=True)
    g = torch.Generator("cpu").manual_seed(sum(shape))
    K, N = shape[-1], 272
    w = (torch.randn(N, K, generator=g) * 0.02).to(torch.bfloat16).cuda()
    b = torch.randn(N, generator=g).to(torch.bfloat16).cuda() if bias else None
    x = torch.randn(shape, generator=g).to(dtype).cuda()
    m = fl.Fp8Linear(w, b, scaling=scaling)
    y = m(x)
    xq, xs = (fl.quantize_rowwise if scaling == "rowwise" else fl.quantize_tensor)(x.reshape(-1, K))
    want = torch.empty(xq.shape[0], N, dtype=torch.bfloat16, device="cuda")
    _lib.fp8_gemm(xq, m.weight_fp8, xs.reshape(-1), m.weight_scale.reshape(-1), b, want)
    torch.cuda.synchronize()
    assert y.dtype == dtype and y.shape == (*shape[:-1], N)
    assert torch.equal(y.reshape(-1, N), want.to(dtype))
    # a column slice is made contiguous, a CPU tensor and another type are refused
    wide = torch.cat([x, x], -1)[..., :K]
    assert torch.equal(m(wide), y)
    with pytest.raises(RuntimeError, match="GPU"):
        m(x.cpu())
    with pytest.raises(ValueError, match="bf16, fp16 or fp32"):
        m(x.double())
