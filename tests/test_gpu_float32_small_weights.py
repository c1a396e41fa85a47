"""GPU test of float32 attention weights below the smallest normal float: they count, as far as a denormal float holds them."""
import math

import pytest
import torch

import test_gpu_parity as TP

pytestmark = pytest.mark.gpu
A = TP.A
SCALE, DEV = TP.SCALE, "cuda"


@pytest.mark.parametrize("s", [2, 40])                       # the diagonal tile alone, and one behind it
@pytest.mark.parametrize("exponent", [-120, -128, -135, -140])
def test_weights_below_the_normal_range(A, s, exponent):
    q, k, v = (torch.zeros(1, 8, s, 64) for _ in range(3))
    q[..., 0] = 30.0
    k[:, :, 1, 0] = exponent * math.log(2) / SCALE / 30.0     # the weight of key 1 against key 0: 2^exponent
    k[:, :, 2:, 0] = -1000.0
    v[:, :, 1] = 1e30
    x = [t.to(DEV).requires_grad_(True) for t in (q, k, v, torch.full((8,), -1e4))]
    o = A.attention(*x, SCALE, None, None)
    d_out = torch.zeros_like(o)
    d_out[:, 1] = 1.0
    dv = torch.autograd.grad(o, x, d_out)[2]
    weight = math.exp(float(q[0, 0, 1, 0]) * float(k[0, 0, 1, 0]) * SCALE)
    # the logit in log2 units is good to a few units of 2^-24 of its size (140), the weight to half of the smallest float
    rel = 4 * 140 * 2.0 ** -24 * math.log(2) + 2.0 ** -150 / weight
    assert bool(((o[0, 1].double().cpu() / 1e30 - weight).abs() <= rel * weight).all())
    assert bool(((dv[0, :, 1].double().cpu() - weight).abs() <= rel * weight).all())
