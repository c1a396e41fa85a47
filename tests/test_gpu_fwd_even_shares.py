"""Chunks of a prompt whose workgroups are more than the compute units, or three quarters of them: shares of the keys that even the rounds out, on both sides
of the rule's lines, against float64 on the GPU."""
import ctypes

import pytest
import torch

from oregon_gpt_oss_patching_amd import _lib, attention_kernel as ak

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("b,h,g,sq,skv,lens,shares", [
    (1, 64, 8, 1024, 6081, None, 1), (1, 64, 8, 1025, 6081, None, 3), (1, 64, 8, 1025, 6080, None, 1),      # 256 and 272 workgroups; 96 tiles, the last of one key, and 95
    (1, 64, 8, 1344, 6100, None, 3), (1, 64, 8, 1345, 6100, None, 2), (1, 64, 8, 1536, 6100, None, 2), (1, 64, 8, 1537, 6100, None, 1),      # 336, 352, 384, 400
    (1, 64, 8, 640, 8129, None, 3), (1, 64, 8, 704, 8129, None, 4), (1, 64, 8, 704, 8128, None, 1), (1, 64, 8, 768, 8129, None, 4), (1, 64, 8, 769, 8129, None, 1),
    (3, 32, 4, 700, 6100, [6100, 5700, 100], 3),
])
def test_shares_that_even_the_rounds_out(b, h, g, sq, skv, lens, shares):
    gen = torch.Generator(device=DEV).manual_seed(skv + sq)
    n = lambda *x: torch.randn(x, generator=gen, device=DEV)
    q, k, v, sinks = n(b, h, sq, 64).bfloat16(), n(b, g, skv, 64).bfloat16(), n(b, skv, g, 64).bfloat16().transpose(1, 2), n(h)
    start = skv - sq
    p = ak._base_params(q, k, v, sinks, None, 0.125, None, start)
    assert _lib.load().gptoss_attn_fwd_workspace_bytes(ctypes.byref(p)) == (shares * b * h * sq * 66 * 4 if shares > 1 else 0)
    o, lse = ak.attention_forward(q, k, v, sinks, 0.125, q_offset=start, seqlens=lens)
    future = torch.arange(skv, device=DEV)[None] > torch.arange(start, skv, device=DEV)[:, None]
    for bi in range(b):
        live = sq if lens is None else max(0, lens[bi] - start)
        for hi in range(0, h, 13):
            logits = (q[bi, hi].double() @ k[bi, hi // (h // g)].double().T * 0.125).masked_fill(future, float("-inf"))
            want_lse = torch.logaddexp(logits.logsumexp(1), sinks[hi].double())
            want = torch.exp(logits - want_lse[:, None]) @ v[bi, hi // (h // g)].double()
            want[live:], want_lse[live:] = 0, sinks[hi].double()
            got = o[bi, :, hi].double()
            # P and O rounded to bf16: 1e-2 relative, 2e-2 absolute plus half an ulp; lse 1e-3
            assert float((got - want).norm()) <= 1e-2 * float(want.norm()) + 1e-30
            assert bool(((got - want).abs() <= 2e-2 + 2.0 ** -8 * want.abs()).all())
            assert float((lse[bi, hi].double() - want_lse).abs().max()) <= 1e-3
