"""attention() where nothing is differentiated takes no autograd node: the same bits as the call that records one, and what the node
refuses or converts stays refused or converted."""
import pytest
import torch
import torch.autograd.forward_ad as fwAD

import oregon_gpt_oss_patching_amd as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("sq,skv,window", [(1, 300, None), (65, 65, 32), (257, 257, None)])
@pytest.mark.parametrize("mode", ["plain", "no_grad", "inference_mode"])
def test_inference_gives_the_bits_of_the_recorded_call(dtype, sq, skv, window, mode):
    g = torch.Generator().manual_seed(skv)
    q, k, v = (torch.randn(2, h, s, 64, generator=g).to("cuda", dtype) for h, s in ((8, sq), (2, skv), (2, skv)))
    sinks = torch.randn(8, generator=g).cuda()
    extra = dict(seqlens=torch.tensor([skv, skv - 7])) if sq == skv and window is None else {}      # int64, on the host
    leaf = q.clone().requires_grad_()
    want = A.attention(leaf, k, v, sinks, 0.125, window, skv - sq, **extra)
    assert want.requires_grad
    with {"plain": torch.enable_grad, "no_grad": torch.no_grad, "inference_mode": torch.inference_mode}[mode]():
        got = A.attention(q if mode == "plain" else leaf, k, v, sinks, 0.125, window, skv - sq, **extra)
    assert not got.requires_grad and got.is_inference() == (mode == "inference_mode")
    assert got.dtype == dtype and torch.equal(got, want)


@pytest.mark.parametrize("which", range(4))
def test_a_tangent_on_any_operand_is_refused(which):
    x = [torch.randn(1, 8, 16, 64), torch.randn(1, 2, 16, 64), torch.randn(1, 2, 16, 64), torch.randn(8)]
    x = [t.cuda() for t in x]
    with torch.no_grad(), fwAD.dual_level():
        x[which] = fwAD.make_dual(x[which], torch.ones_like(x[which]))
        with pytest.raises(RuntimeError):
            A.attention(*x, 0.125, None, None)
