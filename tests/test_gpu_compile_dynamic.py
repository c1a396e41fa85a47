"""GPU tests of torch.compile over lengths and positions that change from call to call: the second call's program serves every later
one, with the eager bits."""
import pytest
import torch

from oracle import eager_ref as E
import test_gpu_parity as TP

pytestmark = pytest.mark.gpu
A = TP.A
SCALE, DEV = TP.SCALE, "cuda"


@pytest.mark.parametrize("dynamic", [True, None])      # None: the first length by itself, then a program for any
@pytest.mark.parametrize("window", [None, 128])
def test_training_over_changing_lengths(A, window, dynamic):
    from torch._dynamo.testing import CompileCounterWithBackend
    torch._dynamo.reset()
    counter = CompileCounterWithBackend("aot_eager")

    def fn(q, k, v, s):
        return A.attention(q, k, v, s, SCALE, window, None)

    compiled = torch.compile(fn, backend=counter, fullgraph=True, dynamic=dynamic)
    programs = []
    for length in (384, 200, 777, 130):
        print(f"case S={length} W={window} dynamic={dynamic}", flush=True)
        *qkvs, d_out = E.make_inputs(9300 + length, 2, 16, 2, length, 64, torch.bfloat16)
        got = []
        for f in (fn, compiled):
            x = [t.to(DEV).requires_grad_(True) for t in qkvs]
            out = f(*x)
            out.backward(d_out.to(DEV))
            got.append([out, *(t.grad for t in x)])
        assert all(torch.equal(a, b) for a, b in zip(*got))
        programs.append(counter.frame_count)
    assert programs[-1] == programs[1]


def test_decoding_at_changing_positions(A):
    from torch._dynamo.testing import CompileCounterWithBackend
    torch._dynamo.reset()
    counter = CompileCounterWithBackend("aot_eager")
    q, k, v, sinks, _ = (t.to(DEV) for t in E.make_inputs(9400, 1, 16, 2, 1, 64, torch.bfloat16, skv=400))

    def fn(keys, values, start):
        return A.attention(q, keys, values, sinks, SCALE, None, start)

    compiled = torch.compile(fn, backend=counter, fullgraph=True)
    programs = []
    with torch.no_grad():
        for n in (300, 301, 350, 399):
            args = (k[:, :, :n], v[:, :, :n], n - 1)
            assert torch.equal(compiled(*args), fn(*args))
            programs.append(counter.frame_count)
    assert programs[-1] == programs[1]
