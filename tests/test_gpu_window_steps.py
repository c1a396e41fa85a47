"""GPU tests of the single-pass window backward's steps: blocks of 32 rows that end anywhere, one pair of heads per block and odd numbers of heads, windows on
and off block edges, chunks whose last one is shorter than a window, against the eager oracle; what padding holds does not reach the rows that exist."""
import pytest
import torch

from oracle import eager_ref as E
import test_gpu_parity as TP

pytestmark = pytest.mark.gpu
A = TP.A
SCALE, DEV = TP.SCALE, "cuda"


@pytest.mark.parametrize("b,h,g,s,w,lens", [
    (1, 4, 2, 31, 16, None),                     # one block that is not full
    (1, 4, 2, 160, 128, None),                   # a step per block
    (2, 6, 2, 129, 128, None),                   # three heads: a step without a head for group 1; a last block of one row
    (1, 5, 1, 353, 97, None),
    (1, 16, 1, 193, 33, None),
    (1, 32, 2, 417, 128, None),                  # sixteen heads; several chunks, the last one of one or two blocks
    (2, 8, 4, 321, 32, [321, 97]),
    (3, 8, 1, 288, 127, [288, 1, 160]),
    (1, 8, 2, 545, 65, None),
    (1, 2, 1, 4001, 128, None),                  # chunks of four blocks
])
def test_window_backward_vs_eager_oracle(A, b, h, g, s, w, lens):
    print(f"case B={b} H={h} G={g} S={s} W={w} lens={lens}", flush=True)
    inp = E.make_inputs(7700 + s, b, h, g, s, 64, torch.bfloat16)
    if lens:
        inp = inp[:4] + (TP.mask_dout(inp[4], lens),)
    got = TP.run_hip(A, *inp, w, 0, lens)
    # (dsinks of a few heads is a cancelling sum: within 1e-2 of the sum of its terms' magnitudes, as the end-to-end sweep asks)
    ref = TP.oracle_eager(*inp, w, 0, lens)
    for name, x, y in zip(("o", "lse", "dq", "dk", "dv"), got, ref):
        if name != "lse":
            # dV and dK sum up to 128 rows x 16 heads of products rounded to bf16 (2^-9 relative): 4.5e-2 at 12 and 16 heads (test_gpu_hard_cases)
            TP.check(name, x, y, atol=4.5e-2 if h // g > 8 else 2e-2)
    o, lse = (t.double().cpu() for t in got[:2])
    terms = torch.exp(inp[3].double().view(1, h, 1) - lse) * (o * inp[4].double()).sum(-1).transpose(1, 2)
    assert bool(((got[5].cpu().double() - ref[5].double()).abs() <= 1e-2 * terms.abs().sum((0, 2))).all())
    again = TP.run_hip(A, *inp, w, 0, lens)
    assert all(torch.equal(x, y) for x, y in zip(got, again))


@pytest.mark.parametrize("s,w,lens", [(320, 128, [96, 256]), (300, 64, [32, 160])])
def test_window_backward_of_padded_rows(A, s, w, lens):
    """NaN in whole blocks of padding changes nothing; the gradients of padded rows are zero."""
    print(f"case S={s} W={w} lens={lens}", flush=True)
    q, k, v, sinks, d_out = (t.to(DEV) for t in E.make_inputs(7800 + s, 2, 8, 1, s, 64, torch.bfloat16))
    got = []
    for value in (0.0, float("nan")):
        x = [t.clone() for t in (q, k, v, d_out)]
        for i, n in enumerate(lens):
            for t in x[:3]:
                t[i, :, n:] = value
            x[3][i, n:] = value
        o, lse = A.attention_forward(*x[:3], sinks, SCALE, w, 0, lens)
        got.append(A.attention_backward(*x[:3], sinks, o, lse, x[3], SCALE, w, 0, lens)[:3])
    for a, b in zip(*got):
        assert torch.equal(a, b)
        for i, n in enumerate(lens):
            assert not b[i, :, n:].any()
