"""GPU test of a start position on the device that the caller moves on between forward and backward."""
import pytest
import torch

from oracle import eager_ref as E
import test_gpu_parity as TP

pytestmark = pytest.mark.gpu
A = TP.A
SCALE, DEV = TP.SCALE, "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_position_moved_on_before_the_backward(A, dtype):
    """An int64 position (what torch's own counters are) is converted once, in the forward: the backward stands where the forward stood."""
    q, k, v, sinks, d_out = (t.to(DEV) for t in E.make_inputs(9500, 1, 8, 2, 40, 64, dtype, skv=200))
    grads = []
    for start in (torch.tensor([100], device=DEV), 100):
        x = [t.clone().requires_grad_(True) for t in (q, k, v, sinks)]
        out = A.attention(*x, SCALE, 64, start)
        if torch.is_tensor(start):
            start += 40
        grads.append(torch.autograd.grad(out, x, d_out))
    for a, b in zip(*grads):
        assert torch.equal(a, b)
