"""GPU test of attn_bwd_dkdv64_kernel's pieces: padded and packed batches whose key blocks are divided by their lengths (more blocks than
a wavefront has lanes, rows of no token or one, walks of one piece and of several)."""
import random

import pytest
import torch

import test_gpu_work_division as TWD

pytestmark = pytest.mark.gpu
A = TWD.A
_check = TWD.test_64_key_backward_of_any_length_vs_eager_oracle


@pytest.mark.parametrize("b,h,g,s,lens,docs", [
    (33, 8, 2, 1030, [1030, 0, 1, 256, 257, 1024] + [random.Random(5).randint(1, 1030) for _ in range(27)], None),
    (2, 8, 1, 2050, [2050, 1], None),                          # one KV head: 256 units for it
    (2, 16, 2, 2560, [2560, 64], [2500, 60]),                  # documents in padded rows
    (1, 8, 4, 2300, None, [1, 1, 2040, 2, 256]),
    (65, 4, 4, 1100, [1 + 17 * i % 1100 for i in range(65)], None),    # one head per KV head
])
def test_pieces_vs_eager_oracle(A, b, h, g, s, lens, docs):
    _check(A, b, h, g, s, lens, docs)


@pytest.mark.parametrize("b,h,g,s", [(7, 8, 8, 1283), (33, 4, 2, 1344)])       # off whole tiles and on them
def test_several_rows_of_one_length(A, b, h, g, s):
    _check(A, b, h, g, s, None, None)
