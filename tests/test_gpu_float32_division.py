"""GPU tests of the float32 kernels' division of work: units of 32 query rows shared by four, two or one wavefronts (the
number of units and the window decide), workgroups whose last units do not exist, key blocks cut into slices."""
import pytest
import torch

from oracle import eager_ref as E
import test_gpu_float32 as TF

pytestmark = pytest.mark.gpu
A = TF.A


@pytest.mark.parametrize("b,h,g,s,w,lens,docs", [
    (1, 8, 2, 97, None, None, None),               # four wavefronts per unit; a last block of one row
    (5, 9, 3, 800, None, None, None),              # 1125 units of a group of three: two wavefronts per unit, an odd count per KV head
    (5, 9, 3, 800, 64, None, None),                # the same with a window: one wavefront per unit, 125 * 3 units in fours
    (5, 9, 3, 800, 700, None, None),               # a long window keeps two
    (3, 16, 2, 737, None, [737, 40, 512], None),   # padded rows in rotation
    (1, 8, 1, 300, None, None, [1, 63, 128, 97, 11]),
    (1, 4, 4, 256, None, None, None),              # one head per KV head: slices of the key blocks
])
def test_float32_vs_eager_oracle(A, b, h, g, s, w, lens, docs):
    print(f"case B={b} H={h} G={g} S={s} W={w} lens={lens} docs={docs}", flush=True)
    q, k, v, sinks, d_out = E.make_inputs(6000 + s + b, b, h, g, s, 64, torch.float32)
    if lens:
        d_out = d_out * (torch.arange(s).view(1, s) < torch.tensor(lens).view(b, 1)).view(b, s, 1, 1)
    ds = E.doc_start_from_lengths([docs] * b, s) if docs else None
    got = TF.run_hip(A, q, k, v, sinks, d_out, w, 0, lens, ds)
    ref = TF.oracle64(q, k, v, sinks, d_out, w, 0, lens, ds)
    for name, x, y in zip(("o", "lse", "dq", "dk", "dv", "dsinks"), got, ref):
        x, y = x.double().cpu(), y.double().cpu()
        # fp32 products and sums of up to a few thousand terms: 2e-5 relative, the float32 path's bound
        assert float((x - y).norm()) <= 2e-5 * float(y.norm()), name
    again = TF.run_hip(A, q, k, v, sinks, d_out, w, 0, lens, ds)
    assert all(torch.equal(x, y) for x, y in zip(got, again))
