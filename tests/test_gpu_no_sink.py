"""GPU tests of sink logits of -inf (no sink: the plain softmax) where a wavefront or a row's first tile holds no key that the row sees:
float32 rows shared by several wavefronts, and the general bf16 forward."""
import pytest
import torch

from oracle import eager_ref as E
import test_gpu_parity as TP

pytestmark = pytest.mark.gpu
A = TP.A
SCALE, DEV = TP.SCALE, "cuda"


def _doc_start(s, docs):
    return torch.tensor([[sum(docs[:i]) for i, n in enumerate(docs) for _ in range(n)]], dtype=torch.int32) if docs else None


def _no_sink(A, dtype, h, g, sq, skv, start, w, docs):
    print(f"case {dtype} H={h} G={g} Sq={sq} Skv={skv} start={start} W={w} docs={docs}", flush=True)
    q, k, v, sinks, d_out = E.make_inputs(9100 + sq + skv, 1, h, g, sq, 64, dtype, skv=skv)
    none = torch.full_like(sinks, float("-inf"))
    ds = _doc_start(sq, docs)
    o, lse = A.attention_forward(*(t.to(DEV) for t in (q, k, v, none)), SCALE, w, start, None, ds)
    f = [t.double() for t in (q, k, v)]
    far = torch.full((h,), -1e4, dtype=torch.float64)       # (exp(-1e4) is 0 beside any logit here: the same softmax)
    args = (far, SCALE, w, start, None, ds)
    return o, lse, E.eager_attention(*f, *args), E.logsumexp_rows(f[0], f[1], *args)


@pytest.mark.parametrize("h,g,sq,skv,start,w,docs", [
    (8, 1, 2, 33, 31, None, None),              # row 0 sees nothing of the second tile, all that the second wavefront walks
    (8, 2, 8, 36, 28, None, None),
    (8, 2, 70, 70, 0, 33, None),                # later rows of a block see nothing of its first tile
    (64, 8, 300, 300, 0, 128, None),            # one wavefront per row block: two tiles in front of some rows' window
    (8, 2, 200, 200, 0, None, [70, 1, 100, 29]),
])
def test_float32_without_sink(A, h, g, sq, skv, start, w, docs):
    o, lse, ref, ref_lse = _no_sink(A, torch.float32, h, g, sq, skv, start, w, docs)
    # the float32 path's bounds: 2e-5 relative (2-norm), lse 2e-5
    assert torch.isfinite(o).all()
    assert float((o.cpu().double() - ref).norm()) <= 2e-5 * float(ref.norm())
    assert float((lse.cpu().double() - ref_lse).abs().max()) <= 2e-5


@pytest.mark.parametrize("h,g,sq,skv,start,w,docs", [
    (8, 2, 300, 300, 0, 100, None),             # a window that is no multiple of 32
    (8, 2, 300, 300, 0, 200, None),
    (6, 2, 200, 200, 0, None, [70, 1, 100, 29]),
    (6, 2, 90, 400, 310, 2000, None),
])
def test_general_forward_without_sink(A, h, g, sq, skv, start, w, docs):
    o, lse, ref, ref_lse = _no_sink(A, torch.bfloat16, h, g, sq, skv, start, w, docs)
    TP.check("o", o, ref.float())
    assert float((lse.cpu().double() - ref_lse).abs().max()) <= TP.LSE_TOL
