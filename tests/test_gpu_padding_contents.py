"""GPU tests of what right-padded rows hold: NaN in the padding of q, k, v and dO changes nothing about the rows that exist."""
import pytest
import torch

from oracle import eager_ref as E
import test_gpu_parity as TP

pytestmark = pytest.mark.gpu
A = TP.A
SCALE, DEV = TP.SCALE, "cuda"


def _padded_with(value, lens, *tensors):
    out = [t.clone() for t in tensors]
    for t in out:
        for b, n in enumerate(lens):
            (t[b, n:] if t is out[-1] else t[b, :, n:]).fill_(value)
    return out


@pytest.mark.parametrize("s,w,lens", [(300, 128, [50, 200]), (321, 64, [300, 97]), (333, 32, [1, 320])])
def test_window_forward_of_padded_rows(A, s, w, lens):
    """O = 0 and lse = sink on padded rows whatever they hold; the sinks' gradient, which runs over all rows, is finite."""
    print(f"case S={s} W={w} lens={lens}", flush=True)
    q, k, v, sinks, d_out = (t.to(DEV) for t in E.make_inputs(9800 + s, 2, 8, 1, s, 64, torch.bfloat16))
    got = []
    for value in (0.0, float("nan")):
        x = _padded_with(value, lens, q, k, v, d_out)
        o, lse = A.attention_forward(*x[:3], sinks, SCALE, w, 0, lens)
        got.append((o, lse))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    for b, n in enumerate(lens):
        assert not got[1][0][b, n:].any()
    x = _padded_with(float("nan"), lens, q, k, v, d_out)
    d_out = _padded_with(0.0, lens, q, k, v, d_out)[-1]
    assert torch.isfinite(A.attention_backward(*x[:3], sinks, o, lse, d_out, SCALE, w, 0, lens)[3]).all()


@pytest.mark.parametrize("s,lens", [(2100, [32, 96]), (2048, [1000, 2047]), (2100, [2100, 64]), (4097, [4000, 130])])
def test_long_rows_dk_dv_of_padded_rows(A, s, lens):
    print(f"case S={s} lens={lens}", flush=True)
    q, k, v, sinks, d_out = (t.to(DEV) for t in E.make_inputs(9900 + s, 2, 8, 1, s, 64, torch.bfloat16))
    got = []
    for value in (0.0, float("nan")):
        x = _padded_with(value, lens, q, k, v, d_out)
        o, lse = A.attention_forward(*_padded_with(0.0, lens, q, k, v, d_out)[:3], sinks, SCALE, None, 0, lens)
        got.append(A.attention_backward(*x[:3], sinks, o, lse, x[3], SCALE, None, 0, lens))
    for a, b in zip(got[0][1:3], got[1][1:3]):             # dK, dV
        for row, n in enumerate(lens):
            assert torch.isfinite(b[row, :, :n]).all() and torch.equal(a[row, :, :n], b[row, :, :n])


@pytest.mark.parametrize("s,w,lens", [(320, None, [200, 97]), (333, 100, [1, 320]), (257, None, [256, 225])])
@pytest.mark.parametrize("value", [float("nan"), 1e30])
def test_float32_padded_rows(A, value, s, w, lens):
    """Also numbers that three bf16 terms do not hold: the rows that exist keep their bits."""
    print(f"case S={s} W={w} lens={lens} value={value}", flush=True)
    q, k, v, sinks, d_out = (t.to(DEV) for t in E.make_inputs(9950 + s, 2, 64, 8, s, 64, torch.float32))
    got = []
    for x in (_padded_with(0.0, lens, q, k, v, d_out), _padded_with(value, lens, q, k, v, d_out)):
        o, lse = A.attention_forward(*x[:3], sinks, SCALE, w, 0, lens)
        got.append((o, lse) + A.attention_backward(*x[:3], sinks, o, lse, x[3], SCALE, w, 0, lens)[:3])
    for a, b in zip(*got):
        assert torch.equal(a, b)
    for b, n in enumerate(lens):
        assert not got[1][0][b, n:].any()
