"""Backward of small problems, dQ and dK/dV in one launch: the bits of the separate entry points, and the oracle, on both sides of every line of the
route (attn_bwd_both_kernel)."""
import pytest
import torch

import oregon_gpt_oss_patching_amd as A
from oracle import eager_ref

pytestmark = pytest.mark.gpu
DEV = "cuda"

# (batch, heads, KV heads, queries, keys, window, valid lengths, documents)
_CASES = [
    (1, 4, 1, 1, 1, None, None, None),                   # one row
    (1, 8, 1, 33, 33, None, None, None),
    (2, 5, 1, 65, 65, None, None, None),                 # a wavefront without a head, a tile of one row
    (1, 16, 2, 128, 128, None, None, None),              # the first pieces
    (2, 12, 2, 383, 383, None, None, None),
    (1, 8, 1, 2047, 2047, None, None, None),             # pieces, and slices in the 64-key kernel's place
    (1, 8, 1, 2048, 2048, None, None, None),
    (1, 8, 2, 2111, 2111, None, None, None),
    (4, 8, 1, 1536, 1536, None, None, None),             # 768 workgroups
    (4, 8, 1, 1600, 1600, None, None, None),             # more: one launch after the other
    (3, 8, 1, 700, 700, None, [700, 64, 1], None),       # padding
    (2, 8, 1, 2100, 2100, None, [2100, 999], None),
    (1, 8, 1, 900, 900, None, None, [1, 63, 500, 336]),  # documents
    (1, 8, 1, 2200, 2200, None, None, [100, 1400, 700]),
    (1, 8, 2, 1024, 1024, None, None, None),             # dQ first: one chunk of heads, a row in front of the line, packed, long rows of two
    (1, 8, 2, 1023, 1023, None, None, None),
    (1, 8, 2, 2600, 2600, None, None, [1000, 1599, 1]),
    (1, 8, 1, 4400, 4400, None, None, None),
    (1, 8, 2, 500, 500, 200, None, None),                # windows the single-pass kernel does not take
    (1, 8, 2, 500, 500, 130, None, [170, 330]),
    (1, 8, 1, 400, 400, 100, None, [250, 150]),
    (1, 8, 2, 100, 450, None, None, None),               # queries behind earlier keys
    (2, 8, 2, 70, 200, 64, None, None),
    (21, 64, 8, 160, 160, None, None, None),             # 1008 workgroups of 64 rows, so dQ has 32-row wavefronts
    (22, 64, 8, 160, 160, None, None, None),             # 1056: 64-row ones, and one launch after the other
    (8, 64, 8, 300, 300, 200, None, None),               # a window: under six rounds of 512 workgroups, and over
    (16, 64, 8, 300, 300, 200, None, None),
    (1, 32, 8, 2048, 2048, None, None, None),            # in the 64-key kernel's place: three rounds
    (1, 32, 8, 2049, 2049, None, None, None),            # 1608
    (2, 8, 2, 1500, 1500, None, [1500, 600], None),      # slices, dQ first
    (4, 16, 2, 700, 700, 200, None, None),
]


# float32 (attn_f32_both_kernel): up to 1024 workgroups, 640 up to 256 rows; key blocks cut into up to sixteen slices, a window's too
_FLOAT32 = [
    (1, 4, 1, 1, 1, None, None, None),
    (1, 3, 1, 31, 31, None, None, None),
    (1, 8, 1, 33, 33, None, None, None),
    (1, 64, 8, 128, 128, None, None, None),              # 384 workgroups
    (2, 64, 8, 129, 129, None, None, None),              # 1040, one launch after the other
    (1, 8, 1, 513, 513, None, None, None),               # sixteen slices
    (1, 2, 2, 700, 700, None, None, None),               # one head per KV head: slices of eight tiles
    (2, 8, 2, 1000, 1000, None, None, None),             # 1024 workgroups
    (1, 8, 1, 400, 400, 128, None, None),                # five tiles see a block
    (2, 6, 1, 300, 300, 33, None, None),
    (1, 8, 1, 1300, 1300, 1299, None, None),
    (3, 8, 1, 400, 400, None, [400, 33, 0], None),
    (2, 8, 2, 300, 300, 100, [300, 170], None),
    (1, 8, 1, 500, 500, None, None, [1, 63, 200, 236]),
    (1, 8, 2, 500, 500, 70, None, [170, 330]),
    (1, 8, 2, 100, 450, None, None, None),               # queries behind earlier keys
    (2, 8, 2, 70, 200, 64, None, None),
]


@pytest.mark.parametrize("dtype,b,h,g,sq,skv,w,lens,docs", [(torch.bfloat16, *c) for c in _CASES] + [(torch.float32, *c) for c in _FLOAT32])
def test_one_launch_against_separate_steps_and_the_oracle(dtype, b, h, g, sq, skv, w, lens, docs):
    gen = torch.Generator().manual_seed(skv + h)
    q, k, v, do = (torch.randn(*n, generator=gen).to(dtype) for n in ((b, h, sq, 64), (b, g, skv, 64), (b, skv, g, 64), (b, sq, h, 64)))
    v = v.transpose(1, 2)
    sinks = torch.randn(h, generator=gen)
    if lens is not None:
        for i, n in enumerate(lens):
            do[i, n:] = 0
    doc_start = None
    if docs is not None:
        doc_start = torch.cat([torch.full((n,), sum(docs[:i]), dtype=torch.int32) for i, n in enumerate(docs)]).view(1, -1)
    start = skv - sq
    dev = [t.to(DEV) for t in (q, k, v, sinks)]
    extra = dict(doc_start=None if doc_start is None else doc_start.to(DEV))
    o, lse = A.attention_forward(*dev, 0.125, w, start, lens, **extra)
    one = A.attention_backward(*dev, o, lse, do.to(DEV), 0.125, w, start, lens, **extra)
    if dtype == torch.float32 or not (w is not None and w <= 128 and docs is None and start == 0):
        three = A.attention_backward(*dev, o, lse, do.to(DEV), 0.125, w, start, lens, split=True, **extra)
        assert all(torch.equal(x, y) for x, y in zip(one, three))
    x = [t.double().requires_grad_() for t in (q, k, v, sinks)]
    eager_ref.eager_attention(*x, 0.125, w, start, lens, doc_start).backward(do.double())
    for name, got, want in zip(("dq", "dk", "dv", "dsinks"), one, x):
        # P, dS and the results rounded to bf16 (2^-9 each, relative): 1e-2 as everywhere; one row's dS is the rounding of O alone.  float32: 2e-5
        got = got.double().cpu()
        assert torch.isfinite(got).all(), name
        rel, one_row = (1e-2, 2e-2) if dtype == torch.bfloat16 else (2e-5, 1e-6)
        assert (got - want.grad).norm() <= rel * want.grad.norm() + (one_row if skv == 1 else 0.0), name
