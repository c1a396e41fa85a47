"""GPU test of a key / value cache whose rows behind the last query hold anything (nobody has written them yet): with the last query at
the end of a 64-key tile the forward kernels read nothing that matters behind it."""
import pytest
import torch

from oracle import eager_ref as E
import test_gpu_parity as TP

pytestmark = pytest.mark.gpu
A = TP.A
SCALE, DEV = TP.SCALE, "cuda"


@pytest.mark.parametrize("sq,start,w", [
    (16, 48, 128), (17, 47, 32), (40, 88, 64), (100, 156, 96), (33, 479, 128),    # window layers, blocks of 32 and 64 rows, tiles' ends
    (16, 48, None), (100, 156, None), (1, 63, None), (1, 63, 128),
])
@pytest.mark.parametrize("lens", [None, 0])
def test_rows_behind_the_last_query_do_not_matter(A, sq, start, w, lens):
    print(f"case Sq={sq} start={start} W={w} lens={lens}", flush=True)
    end = start + sq
    q, k, v, sinks, _ = (t.to(DEV) for t in E.make_inputs(9200 + sq, 1, 8, 1, sq, 64, torch.bfloat16, skv=640))
    lens = None if lens is None else [end]
    off = torch.tensor([start], dtype=torch.int32, device=DEV)
    for on_device in (False, True):
        args = (sinks, SCALE, w, 0 if on_device else start, lens, None, off if on_device else None)
        k[:, :, end:] = 1.0
        v[:, :, end:] = 1.0
        o, lse = A.attention_forward(q, k, v, *args)
        k[:, :, end:] = float("nan")
        v[:, :, end:] = float("nan")
        o2, lse2 = A.attention_forward(q, k, v, *args)
        assert torch.isfinite(o2).all() and torch.equal(o, o2) and torch.equal(lse, lse2)
