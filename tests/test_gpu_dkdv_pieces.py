"""GPU test of attn_bwd_dkdv64_kernel's pieces: padded and packed batches whose key blocks are divided by their lengths (more blocks than
a wavefront has lanes, rows of no token or one, walks of one piece and of several)."""
import ctypes
import random

import pytest
import torch

import test_gpu_work_division as TWD

pytestmark = pytest.mark.gpu
A = TWD.A
_check = TWD.test_64_key_backward_of_any_length_vs_eager_oracle


def _takes_pieces(b, h, g, s, lens, docs):
    """attn_bwd_dkdv64_kernel with room for partial sums behind the row statistics, and a reason to divide by lengths."""
    from oregon_gpt_oss_patching_amd import _lib
    p = _lib.new_params()
    p.B, p.H, p.G, p.Sq, p.Skv, p.D, p.scale = b, h, g, s, s, 64, 0.125
    p.seqlens, p.doc_start = 256 if lens else None, 256 if docs else None
    blocks = b * g * -(-s // 128)
    parts = (_lib.load().gptoss_attn_bwd_workspace_bytes(ctypes.byref(p)) - 24 * b * h * s) // (512 * b * g * s)
    if docs and not lens and h // g <= 4 and b * g * -(-s // 256) * parts <= 256:
        return False                                           # (equal shares that run all at once)
    return parts > 1 and (blocks > 512 or s >= 2048) and bool(lens or docs or (b > 1 and s < 4096 and blocks > 512))


@pytest.mark.parametrize("b,h,g,s,lens,docs", [
    (33, 8, 2, 1030, [1030, 0, 1, 256, 257, 1024] + [random.Random(5).randint(1, 1030) for _ in range(27)], None),
    (2, 8, 1, 2050, [2050, 1], None),                          # one KV head: 256 units for it
    (2, 16, 2, 2560, [2560, 64], [2500, 60]),                  # documents in padded rows
    (1, 8, 4, 2300, None, [1, 1, 2040, 2, 256]),
    (40, 4, 4, 1100, [1 + 27 * i % 1100 for i in range(40)], None),    # one head per KV head
    # the most key blocks of a KV head.  (64 tokens at least: dQ of a row of one is dS = P (dP - delta) = P (1 - P) dP times K, and delta's O is rounded to bf16, which
    # moves it by 2^-9 P / (1 - P), 0.8 % at P = 0.8, before dS and dQ are rounded)
    (227, 1, 1, 1030, [64 + 37 * i % 967 for i in range(227)], None),
])
def test_pieces_vs_eager_oracle(A, b, h, g, s, lens, docs):
    assert _takes_pieces(b, h, g, s, lens, docs)
    _check(A, b, h, g, s, lens, docs)


def test_too_many_rows_for_pieces(A):
    lens = [1 + 17 * i % 1100 for i in range(65)]
    assert not _takes_pieces(65, 4, 4, 1100, lens, None)
    _check(A, 65, 4, 4, 1100, lens, None)


@pytest.mark.parametrize("b,h,g,s", [(7, 8, 8, 1283), (33, 4, 2, 1344)])       # off whole tiles and on them
def test_several_rows_of_one_length(A, b, h, g, s):
    assert _takes_pieces(b, h, g, s, None, None)
    _check(A, b, h, g, s, None, None)


@pytest.mark.parametrize("b,h,g,s,docs", [(1, 8, 2, 2300, [1, 1, 2040, 2, 256]), (1, 16, 4, 2048, [300] * 6 + [248]), (2, 8, 2, 2048, [100] * 20 + [48])])
def test_packed_rows_of_few_heads_in_equal_shares(A, b, h, g, s, docs):
    assert not _takes_pieces(b, h, g, s, None, docs)
    _check(A, b, h, g, s, None, docs)
