"""dK/dV of one or several short rows, cut into pieces of (query tile, head) steps that start and end inside a tile."""
import pytest
import torch

import oregon_gpt_oss_patching_amd as A
from oracle import eager_ref

pytestmark = pytest.mark.gpu


def _piece_steps(b, h, g, s):
    """What dkdv_parts_for and dkdv_pieces_for decide for rows of one length below 2048 tokens: steps of a piece, 0 where slices of whole tiles stay."""
    up = lambda n, d: -(-n // d)
    blocks, tiles, r = up(s, 128), up(s, 64), h // g
    n = g * b * blocks
    parts = up(768 if s <= 1024 else 1024, n) if n <= 512 else (2 if b > 1 and s >= 1280 and n < 1024 else 1)
    parts = max(1, min(parts, tiles * r // 8, tiles, 8))
    most = min(parts * s // 128, 512 // (g * b))
    if parts == 1 or most < blocks:
        return 0
    total = blocks * (tiles + 1 - blocks) * r
    for steps in range(up(total, most) if total > 4 * most else 4, up(tiles, parts) * r + (b == 1)):
        if sum(up((tiles - 2 * i) * r, steps) for i in range(blocks)) <= most:
            return steps
    return 0


# the smallest rows that take pieces, ends of tiles and of key blocks, the last row in front of the 64-key kernel, group sizes that a piece does not
# divide, one head per KV head, three rows and more
_PIECES = [(1, 8, 1, 128), (1, 8, 1, 171), (2, 16, 2, 383), (1, 8, 1, 1024), (1, 8, 1, 1023), (1, 5, 1, 700), (2, 6, 2, 448), (1, 16, 1, 640), (1, 8, 1, 2047),
           (1, 4, 4, 961), (1, 8, 8, 2047), (2, 4, 4, 1027), (3, 8, 2, 385), (4, 16, 1, 1999), (8, 8, 1, 309), (5, 6, 2, 1342)]
# slices of whole tiles, and a row that is not cut
_SLICES = [(1, 8, 1, 65), (1, 16, 2, 129), (3, 8, 2, 257), (1, 4, 4, 900), (8, 8, 1, 300)]


@pytest.mark.parametrize("b,h,g,s,pieces", [c + (True,) for c in _PIECES] + [c + (False,) for c in _SLICES])
def test_short_rows_against_the_oracle(b, h, g, s, pieces):
    assert (_piece_steps(b, h, g, s) > 0) == pieces
    _check(b, h, g, s)


def _check(b, h, g, s):
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
