"""The LayerNorm that quantises its own rows against the LayerNorm and the row-wise
quantiser one after the other: the residual stream, the codes and the scales bit for
bit, over row lengths at the edges of a wavefront's registers."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K", [(1, 8), (5, 504), (9, 520), (8195, 264), (130, 3072), (3, 4096)])
@pytest.mark.parametrize("res", [False, True], ids=["plain", "residual"])
@pytest.mark.parametrize("affine,mod", [(False, True), (True, False), (True, True), (False, False)])
def test_ln_quant_equals_the_two_passes(M, K, res, affine, mod):
    from sr_dit import _lib
    print(f"[case] ln_quant M={M} K={K} res={res} affine={affine} mod={mod}", flush=True)
    g = torch.Generator("cpu").manual_seed(M + K)

    def rows(ld):
        t = torch.full((M, ld), 1e3, dtype=torch.bfloat16)
        t[:, :K] = torch.randn(M, K, generator=g).to(torch.bfloat16)
        return t.cuda()[:, :K]

    def vec(dtype, mean=0.0):
        return (torch.randn(K, generator=g) * 0.3 + mean).to(dtype).cuda()

    x, y = rows(K + 8), rows(K + 16)
    x[0] = 2.0                                       # a constant row: LayerNorm 0
    if M > 4:
        x[3, K // 2] = float("inf")                  # its row becomes NaN, the others do not
    gate = vec(torch.float32)
    w, b = (vec(torch.bfloat16, 1.0), vec(torch.bfloat16)) if affine else (None, None)
    sc, sh = (vec(torch.float32), vec(torch.float32)) if mod else (None, None)
    out = torch.empty(M, K, dtype=torch.bfloat16, device="cuda")
    want_x = torch.empty_like(out)
    if res:
        _lib.residual_ln_modulate(x, y, gate, want_x, w, b, sc, sh, 1e-6, out)
    else:
        _lib.ln_modulate(x, w, b, sc, sh, 1e-6, out)
    f8 = torch.float8_e4m3fn
    want_q, want_s = torch.empty(M, K, dtype=f8, device="cuda"), torch.empty(M, device="cuda")
    _lib.fp8_quant_rowwise(out, want_q, want_s)
    got_x = torch.empty_like(out)
    got_q, got_s = torch.empty_like(want_q), torch.empty_like(want_s)
    _lib.residual_ln_quant(x, y if res else None, gate if res else None, got_x if res else None, w,
                           b, sc, sh, 1e-6, got_q, got_s)
    torch.cuda.synchronize()
    assert torch.equal(got_q.view(torch.uint8), want_q.view(torch.uint8))
    assert torch.equal(got_s.view(torch.int32), want_s.view(torch.int32))
    if res:
        assert torch.equal(got_x.view(torch.int16), want_x.view(torch.int16))
