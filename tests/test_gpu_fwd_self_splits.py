"""Self-attention on few heads, whose forward cuts the keys of every query block into shares: on both sides of the rule's lines and at the ends of tiles, padded
rows and sharply rising logits among them, against float64 on the GPU."""
import ctypes

import pytest
import torch

from oregon_gpt_oss_patching_amd import _lib, attention_kernel as ak

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("b,h,g,s,lens,shares", [
    (1, 4, 1, 1217, None, 2),                   # 20 tiles, the last of one key
    (1, 8, 1, 1216, None, 1), (2, 8, 1, 1279, None, 2), (1, 8, 1, 2047, None, 4), (1, 4, 1, 2048, None, 4), (1, 12, 3, 1601, None, 3), (1, 16, 2, 2496, None, 3),
    (3, 8, 1, 1601, None, 1), (1, 20, 1, 1601, None, 1),      # six groups of four heads, five
    (2, 8, 1, 8128, None, 1), (1, 8, 1, 8128, None, 2),       # 127 tiles: 508 workgroups, 254
    (2, 8, 1, 8129, None, 2), (2, 8, 1, 8193, None, 1), (1, 8, 1, 8129, None, 4), (1, 4, 1, 8129, None, 8),      # 128
    (1, 8, 1, 16384, None, 2),
    (3, 4, 1, 1600, [1600, 777, 0], 3),
    (2, 8, 1, 2497, [2497, 1], 3),
])
@pytest.mark.parametrize("lift", [0.0, 40.0])
def test_shares_of_self_attention(b, h, g, s, lens, shares, lift):
    gen = torch.Generator(device=DEV).manual_seed(s + h)
    n = lambda *x: torch.randn(x, generator=gen, device=DEV)
    q, k, v, sinks = n(b, h, s, 64).bfloat16(), n(b, g, s, 64).bfloat16(), n(b, s, g, 64).bfloat16().transpose(1, 2), n(h)
    if lift:
        k[:, :, s // 2:] *= lift
    p = ak._base_params(q, k, v, sinks, None, 0.125, None, 0)
    assert _lib.load().gptoss_attn_fwd_workspace_bytes(ctypes.byref(p)) == (shares * b * h * s * 66 * 4 if shares > 1 else 0)
    o, lse = ak.attention_forward(q, k, v, sinks, 0.125, seqlens=lens)
    again = ak.attention_forward(q, k, v, sinks, 0.125, seqlens=lens)
    assert torch.equal(o, again[0]) and torch.equal(lse, again[1])
    causal = torch.ones(s, s, dtype=torch.bool, device=DEV).triu(1)
    for bi in range(b):
        live = s if lens is None else lens[bi]
        for hi in range(0, h, 3):
            logits = (q[bi, hi].double() @ k[bi, hi // (h // g)].double().T * 0.125).masked_fill(causal, float("-inf"))
            want_lse = torch.logaddexp(logits.logsumexp(1), sinks[hi].double())
            want = torch.exp(logits - want_lse[:, None]) @ v[bi, hi // (h // g)].double()
            want[live:], want_lse[live:] = 0, sinks[hi].double()
            got = o[bi, :, hi].double()
            # P and O rounded to bf16: 1e-2 relative, 2e-2 absolute plus half an ulp; lse 1e-3, with lifted keys the fp32 rounding of logits of order 300
            assert float((got - want).norm()) <= 1e-2 * float(want.norm()) + 1e-30
            assert bool(((got - want).abs() <= 2e-2 + 2.0 ** -8 * want.abs()).all())
            assert float((lse[bi, hi].double() - want_lse).abs().max()) <= 1e-3 * (1 + (float(want_lse.abs().max()) / 64 if lift else 0))
