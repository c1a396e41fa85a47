"""GPU tests of the one-pass window forward off whole 32-row blocks: any length, query offsets (by value and on the device), padded
rows, packed documents, caches that end before or behind the queries, against the eager oracle; and against
attn_fwd_kernel, which a window that is no multiple of 32 takes."""
import pytest
import torch

from oracle import eager_ref as E
import test_gpu_parity as TP

pytestmark = pytest.mark.gpu
A = TP.A
SCALE, DEV = TP.SCALE, "cuda"


@pytest.mark.parametrize("b,h,g,sq,skv,start,lens,docs", [
    (1, 8, 2, 33, 33, 0, None, None),                    # a second block of one row
    (2, 8, 2, 95, 95, 0, None, None),
    (1, 16, 2, 129, 129, 0, None, None),
    (3, 8, 2, 333, 333, 0, [333, 64, 1], None),          # padded rows of a ragged batch
    (1, 16, 2, 200, 1000, 800, None, None),              # a chunk at the end of a cache
    (1, 16, 2, 200, 1000, 333, None, None),              # ... in its middle, not on a block's edge
    (1, 16, 2, 64, 70, 6, None, None),                   # the first rows' windows reach in front of key 0
    (1, 8, 1, 100, 90, 10, None, None),                  # fewer keys than positions
    (1, 8, 1, 100, 40, 10, None, None),                  # ... whole blocks of rows with few keys left, or none
    (2, 8, 2, 100, 600, 500, [600, 520], None),          # padded rows behind an offset
    (1, 8, 2, 514, 514, 0, None, [63, 129, 1, 255, 64, 2]),
    (2, 8, 2, 700, 700, 0, None, [32, 32, 96, 200, 340]),
    (1, 8, 1, 96, 96, 0, None, [1] * 96),
    (2, 8, 2, 500, 500, 0, [500, 300], [290, 10, 200]),  # packed and padded
])
@pytest.mark.parametrize("w", [32, 64, 96, 128])
@pytest.mark.parametrize("on_device", [False, True])
def test_window_forward_of_any_shape_vs_eager_oracle(A, b, h, g, sq, skv, start, lens, docs, w, on_device):
    if on_device and docs:
        pytest.skip("packed rows take no query offset")
    print(f"case B={b} H={h} G={g} Sq={sq} Skv={skv} start={start} lens={lens} docs={docs} W={w} on_device={on_device}", flush=True)
    q, k, v, sinks, _ = E.make_inputs(6000 + sq + skv, b, h, g, sq, 64, torch.bfloat16, skv=skv)
    ds = E.doc_start_from_lengths([docs] * b, sq) if docs else None
    # V as a transposed view of (B, S, G, D), as a model hands it over
    vd = v.transpose(1, 2).contiguous().to(DEV).transpose(1, 2)
    off = torch.tensor([start], dtype=torch.int32, device=DEV) if on_device else None
    o, lse = A.attention_forward(q.to(DEV), k.to(DEV), vd, sinks.to(DEV), SCALE, w, 0 if on_device else start, lens, ds, off)
    f = [t.float() for t in (q, k, v, sinks)]
    TP.check("o", o, E.eager_attention(*f, SCALE, w, start, lens, ds))
    ref = E.logsumexp_rows(f[0], f[1], f[3], SCALE, w, start, lens, ds).float()
    assert float((lse.cpu() - ref).abs().max()) <= TP.LSE_TOL


@pytest.mark.parametrize("sq", [64 * 128 + 1, 64 * 128 + 32, 64 * 128 + 63])
def test_pairs_of_blocks_end_anywhere(A, sq):
    """Enough blocks that a workgroup takes two of them; the last pair is short."""
    print(f"case S={sq}", flush=True)
    q, k, v, sinks, _ = (t.to(DEV) for t in E.make_inputs(6100, 1, 64, 8, sq, 64, torch.bfloat16))
    o, lse = A.attention_forward(q, k, v, sinks, SCALE, 128)
    tail = slice(sq - 200, sq)
    f = [t.float().cpu() for t in (q[:, :, tail], k[:, :, sq - 400:], v[:, :, sq - 400:], sinks)]
    TP.check("o", o[:, tail], E.eager_attention(*f, SCALE, 128, 200))
    assert float((lse[:, :, tail].cpu() - E.logsumexp_rows(f[0], f[1], f[3], SCALE, 128, 200).float()).abs().max()) <= TP.LSE_TOL
