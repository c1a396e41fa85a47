"""GPU test of packed rows whose documents start at multiples of 64: what one document holds (NaN) does not reach another's forward."""
import pytest
import torch

from oracle import eager_ref as E
import test_gpu_parity as TP

pytestmark = pytest.mark.gpu
A = TP.A
SCALE, DEV = TP.SCALE, "cuda"


@pytest.mark.parametrize("w", [None, 32, 128, 100])
@pytest.mark.parametrize("docs", [(64, 128, 64), (512, 1024, 701), (128, 256, 1664)])
def test_documents_keep_their_nans(A, docs, w):
    print(f"case docs={docs} W={w}", flush=True)
    s = sum(docs)
    q, k, v, sinks, _ = (t.to(DEV) for t in E.make_inputs(9990 + s, 1, 8, 1, s, 64, torch.bfloat16))
    ds = torch.tensor([[sum(docs[:i]) for i, n in enumerate(docs) for _ in range(n)]], dtype=torch.int32, device=DEV)
    o, lse = A.attention_forward(q, k, v, sinks, SCALE, w, 0, None, ds)
    for d in range(len(docs)):
        x = [t.clone() for t in (q, k, v)]
        here = slice(sum(docs[:d]), sum(docs[:d + 1]))
        for t in x:
            t[:, :, here] = float("nan")
        o2, lse2 = A.attention_forward(*x, sinks, SCALE, w, 0, None, ds)
        other = torch.ones(s, dtype=torch.bool, device=DEV)
        other[here] = False
        # (a workgroup that met a NaN may repeat its rows with another softmax reference: two roundings of O, the last places of lse)
        a, b = o2[:, other].float(), o[:, other].float()
        assert torch.isfinite(a).all() and bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + 2.0 ** -9).all())
        assert float((lse2[:, :, other] - lse[:, :, other]).abs().max()) <= 1e-5
