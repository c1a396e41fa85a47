"""Function transforms over attention() are refused, in words (the autograd node has no rules for them)."""
import pytest
import torch

import oregon_gpt_oss_patching_amd as A


def test_vmap_is_refused_rather_than_run_slice_by_slice():
    q, k, s = torch.randn(3, 1, 8, 16, 64), torch.randn(3, 1, 2, 16, 64), torch.randn(8)
    with pytest.raises(RuntimeError, match="cannot be vmapped"):
        torch.vmap(lambda a, b: A.attention(a, b, b, s, 0.125, None, None))(q, k)


@pytest.mark.gpu
def test_transforms_are_refused_on_the_gpu():
    q, k, s = (t.to("cuda") for t in (torch.randn(3, 1, 8, 16, 64), torch.randn(3, 1, 2, 16, 64), torch.randn(8)))

    def f(a, b):
        return A.attention(a, b, b, s, 0.125, None, None)

    for call in (lambda: torch.vmap(f)(q, k), lambda: torch.func.grad(lambda a: f(a, k[0]).sum())(q[0]),
                 lambda: torch.func.jvp(lambda a: f(a, k[0]), (q[0],), (q[0],))):
        with pytest.raises(RuntimeError):
            call()
    assert f(q[0], k[0]).shape == (1, 16, 8, 64)
