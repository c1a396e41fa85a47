"""GPU test of sliding-window layers whose softmax scale is next to nothing: the weights are those of equal logits, and dV and dSinks follow from them."""
import pytest
import torch

import oregon_gpt_oss_patching_amd as A

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("scale", [2.0 ** -112, 2.0 ** -118, 1e-38, 2.0 ** -130])
@pytest.mark.parametrize("h,g,s,w", [(8, 2, 200, 128), (5, 1, 161, 64)])
def test_backward_at_the_smallest_scales(scale, h, g, s, w):
    gen = torch.Generator().manual_seed(s)
    q, k, v, do = (torch.randn(*n, generator=gen).bfloat16() for n in ((1, h, s, 64), (1, g, s, 64), (1, g, s, 64), (1, s, h, 64)))
    sinks = torch.randn(h, generator=gen)
    dev = [t.to(DEV) for t in (q, k, v, sinks)]
    o, lse = A.attention_forward(*dev, scale, w)
    dq, dk, dv, dsinks = A.attention_backward(*dev, o, lse, do.to(DEV), scale, w)
    i = torch.arange(s)
    seen = ((i[None] <= i[:, None]) & (i[None] > i[:, None] - w)).double()
    want_dv, want_ds = torch.zeros(g, s, 64, dtype=torch.float64), torch.zeros(h, dtype=torch.float64)
    for hi in range(h):
        z = seen.sum(1, keepdim=True) + sinks[hi].double().exp()
        p = seen / z
        d = do[0, :, hi].double()
        want_dv[hi // (h // g)] += p.T @ d
        want_ds[hi] = -((sinks[hi].double().exp() / z) * ((p @ v[0, hi // (h // g)].double()) * d).sum(1, keepdim=True)).sum()
    assert torch.isfinite(dq).all() and torch.isfinite(dk).all()
    # P, dO and dV in bf16 (2^-9 each, relative): 1e-2; dSinks sums terms of either sign, whose O is rounded to bf16
    assert float((dv[0].double().cpu() - want_dv).norm()) <= 1e-2 * float(want_dv.norm())
    assert float((dsinks.double().cpu() - want_ds).abs().max()) <= 2e-2
