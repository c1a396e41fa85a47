"""GPU tests of the forward's scratch: it is an argument of its own, the block's `delta` belongs to the backward."""
import ctypes

import pytest
import torch

from oracle import eager_ref as E
import test_gpu_parity as TP

pytestmark = pytest.mark.gpu
A = TP.A
SCALE, DEV = TP.SCALE, "cuda"


@pytest.mark.parametrize("sq,skv", [(1, 2049), (100, 2500)])      # decoding slices, shares of the pipelined forward
def test_forward_leaves_delta_alone_and_takes_scratch_of_its_own(A, sq, skv):
    from oregon_gpt_oss_patching_amd import _lib
    from oregon_gpt_oss_patching_amd import attention_kernel as ak
    q, k, v, sinks, _ = (t.to(DEV) for t in E.make_inputs(9600 + sq, 1, 16, 2, sq, 64, torch.bfloat16, skv=skv))
    s32 = sinks.float().contiguous()
    whole, whole_lse = A.attention_forward(q, k, v, s32, SCALE, None, skv - sq)
    p = ak._base_params(q, k, v, s32, None, SCALE, None, skv - sq)
    o, lse = torch.empty_like(whole), torch.empty_like(whole_lse)
    p.o, p.lse = o.data_ptr(), lse.data_ptr()
    ak._set(p.o_stride, ak._strides_bhs(o, "bshd"))
    need = _lib.load().gptoss_attn_fwd_workspace_bytes(ctypes.byref(p))
    assert need > 0
    stream = torch.cuda.current_stream().cuda_stream
    others = torch.full((need // 4 + 64,), 7.0, device=DEV)           # a backward's scratch that is still in use

    def run(name, *between):
        o.fill_(float("nan"))
        lse.fill_(float("nan"))
        _lib.call(name, p, stream, *between)
        torch.cuda.synchronize()
        return o.clone(), lse.clone()

    uncut = run("gptoss_attn_fwd")
    for base in (others.data_ptr(), others.data_ptr() + 4):            # (the forward does not care how it is aligned)
        p.delta = base
        for call in (("gptoss_attn_fwd",), ("gptoss_attn_fwd_sinks", _lib.DTYPE_FP32)):
            assert all(torch.equal(x, y) for x, y in zip(run(*call), uncut))
    mine = torch.empty((need // 4,), device=DEV)
    for size, expect in ((need, (whole, whole_lse)), (need - 16, uncut), (0, uncut)):
        got = run("gptoss_attn_fwd_scratch", _lib.DTYPE_FP32, mine.data_ptr(), size)
        assert all(torch.equal(x, y) for x, y in zip(got, expect))
    assert all(torch.equal(x, y) for x, y in zip(run("gptoss_attn_fwd_scratch", _lib.DTYPE_FP32, None, need), uncut))
    with pytest.raises(_lib.GptossAttnError) as e:
        _lib.call("gptoss_attn_fwd_scratch", p, stream, _lib.DTYPE_FP32, mine.data_ptr() + 4, need)
    assert e.value.status == -7
    assert bool((others == 7.0).all())
    assert float((uncut[0].float() - whole.float()).abs().max()) <= 2.0 ** -6 and float((uncut[1] - whole_lse).abs().max()) <= 1e-5
