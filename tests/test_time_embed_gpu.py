"""The fused time embedding against the chain it replaces (the same sums, so equal up to
the fp32 rounding of the sinusoid and the silu) and against float64."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

U32 = 2.0 ** -24


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("dim,freq,bias", [(8, 8, True), (24, 264, False), (520, 256, True),
                                           (3072, 256, True)])
@pytest.mark.parametrize("t", [0.0, 625.0, 999.75])
def test_time_embed_matches_the_chain(dim, freq, bias, dtype, t):
    from sr_dit import _lib
    from sr_dit.model import sinusoidal_embedding_1d
    print(f"[case] time_embed dim={dim} freq={freq} t={t} {dtype}", flush=True)
    g = torch.Generator("cpu").manual_seed(dim)
    lins = []
    for n, k in ((dim, freq), (dim, dim), (6 * dim, dim)):
        m = torch.nn.Linear(k, n, bias=bias)
        with torch.no_grad():
            m.weight.copy_(torch.randn(n, k, generator=g) / k ** 0.5)
            if bias:
                m.bias.copy_(torch.randn(n, generator=g) * 0.1)
        lins.append(m.to(dtype).cuda())
    tt = torch.tensor([t], device="cuda")
    with torch.no_grad():
        assert _lib.time_embed_fits(tt, lins)
        e, e0 = _lib.time_embed(tt, lins)

        def step(m, x):     # the chain's Linear
            out = torch.empty(1, m.out_features, device="cuda")
            _lib.gemv_f32(x.contiguous(), m.weight, m.bias, out)
            return out

        silu = torch.nn.functional.silu
        x = sinusoidal_embedding_1d(freq, tt).float()
        ce = step(lins[1], silu(step(lins[0], x)))
        ce0 = step(lins[2], silu(ce))

        def exact(m, x):
            y = torch.matmul(x, m.weight.double().T.contiguous())
            return y if m.bias is None else y + m.bias.double()

        xe = exact(lins[1], silu(exact(lins[0], x.double())))
        xe0 = exact(lins[2], silu(xe))
    torch.cuda.synchronize()
    # an ulp of the sinusoid or the silu, carried through a K-term sum
    for got, chain, ref in ((e, ce, xe), (e0, ce0, xe0)):
        scale = ref.norm()
        assert (got.double() - ref).norm() <= 16 * U32 * scale
        assert (got - chain).double().norm() <= 4 * U32 * scale
    # a timestep of another type takes the chain
    assert not _lib.time_embed_fits(tt.double(), lins)
