"""dK/dV of one or several short rows, cut into pieces of (query tile, head) steps that start and end inside a tile."""
import pytest
import torch

import oregon_gpt_oss_patching_amd as A
from oracle import eager_ref

pytestmark = pytest.mark.gpu


# the smallest row that is cut, ends of tiles and of key blocks, the last row in front of the 64-key kernel, group sizes that a piece does not divide
@pytest.mark.parametrize("b,h,g,s", [(1, 8, 1, 65), (1, 8, 1, 128), (1, 16, 2, 129), (2, 16, 2, 383), (1, 8, 1, 1024), (1, 8, 1, 1023),
                                     (3, 8, 2, 257), (1, 5, 1, 700), (2, 6, 2, 448), (1, 4, 4, 900), (1, 16, 1, 640), (1, 8, 1, 2047), (8, 8, 1, 300)])
def test_short_rows_against_the_oracle(b, h, g, s):
    gen = torch.Generator().manual_seed(s + h)
    q, k, v, do = (torch.randn(*n, generator=gen).bfloat16() for n in ((b, h, s, 64), (b, g, s, 64), (b, g, s, 64), (b, s, h, 64)))
    sinks = torch.randn(h, generator=gen)

    def grads(dev, f):
        x = [t.to(dev) if dev == "cuda" else t.double() for t in (q, k, v, sinks)]
        x = [t.requires_grad_() for t in x]
        f(*x).backward(do.to(dev) if dev == "cuda" else do.double())
        return [t.grad.double().cpu() for t in x]

    got = grads("cuda", lambda q, k, v, sk: A.attention(q, k, v, sk, 0.125, None, None))
    again = grads("cuda", lambda q, k, v, sk: A.attention(q, k, v, sk, 0.125, None, None))
    assert all(torch.equal(x, y) for x, y in zip(got, again))
    want = grads("cpu", lambda q, k, v, sk: eager_ref.eager_attention(q, k, v, sk, 0.125))
    for name, x, y in zip(("dq", "dk", "dv", "dsinks"), got, want):
        # P, dS and the results rounded to bf16 (2^-9 each, relative): 1e-2 as everywhere
        assert (x - y).norm() <= 1e-2 * y.norm(), name
