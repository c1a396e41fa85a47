"""GPU tests of library calls that are refused on the host: GptossAttnError with its status, from every way to the operators.  (Nothing is launched.)"""
import pytest
import torch

import test_gpu_parity as TP

pytestmark = pytest.mark.gpu
A = TP.A
SCALE, DEV = TP.SCALE, "cuda"


def _inputs(d=64, grad=False):
    q, k, v = (torch.zeros(1, h, 64, d, dtype=torch.bfloat16, device=DEV, requires_grad=grad) for h in (4, 2, 2))
    return q, k, v, torch.zeros(4, device=DEV, requires_grad=grad)


def test_calls_operators_and_compiled_programs(A):
    from oregon_gpt_oss_patching_amd import _lib
    args = (*_inputs(32), SCALE, 0)
    lse, o = torch.zeros(1, 4, 64, device=DEV), torch.zeros(1, 64, 4, 32, dtype=torch.bfloat16, device=DEV)
    compiled = torch.compile(lambda *x: A.attention(*x, None), backend="aot_eager", fullgraph=True)
    for call in (lambda: A.attention(*args, None), lambda: torch.ops.gptoss_attn.fwd(*args, 0, None, None), lambda: compiled(*args),
                 lambda: torch.ops.gptoss_attn.bwd(*args[:4], o, lse, o, SCALE, 0, 0, None, None, True),
                 lambda: A.attention_forward(*args)):
        with pytest.raises(_lib.GptossAttnError, match="head_dim must be 64") as e:
            call()
        assert e.value.status == -3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_backward(A, dtype):
    """dO that is contiguous but starts between two 16-byte boundaries: refused by the library in the backward."""
    from oregon_gpt_oss_patching_amd import _lib
    q, k, v, sinks = _inputs(grad=True)
    out = A.attention(q.to(dtype), k.to(dtype), v.to(dtype), sinks, SCALE, None, None)
    d_out = torch.zeros(out.numel() + 1, dtype=dtype, device=DEV)[1:].view(out.shape)
    with pytest.raises(_lib.GptossAttnError, match="16-byte aligned") as e:
        out.backward(d_out)
    assert e.value.status == -7
    out.sum().backward()                       # the process goes on
    torch.cuda.synchronize()
