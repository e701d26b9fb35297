"""The row-wise quantiser at the edges of its row lengths: rows held by one
wavefront (up to 4096 elements), by a workgroup (up to 16384) and re-read (longer),
against the oracle's codes and scales bit for bit."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import fp8 as of

pytestmark = pytest.mark.gpu

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


@pytest.mark.parametrize("K", [8, 504, 520, 4096, 4104, 14336, 16384, 16392])
@pytest.mark.parametrize("dtype", sorted(DTYPES))
def test_quant_rowwise_row_lengths(K, dtype):
    from sr_dit import _lib
    print(f"quant_rowwise K={K} {dtype}", flush=True)
    g = torch.Generator("cpu").manual_seed(K)
    M, ldx = 5, K + 8                               # strided rows, a partial last workgroup
    x = torch.zeros(M, ldx)
    x[:, :K] = torch.randn(M, K, generator=g) * 3.0
    x[1] = 0.0                                      # an all-zero row: the scale's floor
    x[2, K - 1] = 40.0                              # the largest value in the row's last chunk
    x[:, K:] = 1e4                                  # past the row: must not count
    x = x.to(DTYPES[dtype])
    q_ref, s_ref = of.quantize_rowwise(x[:, :K].float().numpy())
    q = torch.full((M, K), 0x55, dtype=torch.uint8, device="cuda").view(torch.float8_e4m3fn)
    s = torch.full((M,), -1.0, device="cuda")
    _lib.fp8_quant_rowwise(x.cuda()[:, :K], q, s)
    torch.cuda.synchronize()
    assert np.array_equal(q.view(torch.uint8).cpu().numpy(), q_ref)
    assert np.array_equal(s.cpu().numpy(), s_ref)


@pytest.mark.parametrize("K", [3072, 14336])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_quant_rowwise_non_finite_row_stays_in_its_row(K, bad):
    """A row with an infinity or a NaN takes the true division; its neighbours keep
    their codes, and the NaN or infinite scale is the row's alone."""
    from sr_dit import _lib
    print(f"quant_rowwise K={K} {bad}", flush=True)
    x = torch.randn(4, K, generator=torch.Generator("cpu").manual_seed(K)).to(torch.bfloat16)
    q_ref, s_ref = of.quantize_rowwise(x.float().numpy())
    x[2, 7] = bad
    q = torch.empty((4, K), dtype=torch.float8_e4m3fn, device="cuda")
    s = torch.empty(4, device="cuda")
    _lib.fp8_quant_rowwise(x.cuda(), q, s)
    torch.cuda.synchronize()
    keep = [0, 1, 3]
    assert np.array_equal(q.view(torch.uint8).cpu().numpy()[keep], q_ref[keep])
    assert np.array_equal(s.cpu().numpy()[keep], s_ref[keep])
    assert not torch.isfinite(s[2]).item()
    assert (q.view(torch.uint8)[2, 7].item() & 0x7f) == 0x7f      # NaN code: inf / inf, NaN / NaN
