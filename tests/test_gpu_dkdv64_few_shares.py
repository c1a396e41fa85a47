"""dK/dV of rows of one length on few heads, whose walks are divided by their lengths in the 64-key kernel: against whole key blocks (the backward without
scratch), at the ends of tiles and blocks and on both sides of the line between the divisions."""
import pytest
import torch

from oregon_gpt_oss_patching_amd import _lib, attention_kernel as ak

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("b,h,g,s", [
    (1, 8, 1, 5120), (1, 8, 1, 5121), (1, 8, 1, 5183), (1, 8, 1, 5377),      # whole blocks; a key, a tile less a key, a block and a key more
    (1, 6, 1, 6000), (1, 1, 1, 4100), (1, 16, 1, 4097), (1, 8, 2, 4160), (3, 4, 1, 3000), (1, 32, 4, 2304),
    (1, 32, 4, 2560), (1, 32, 4, 2561), (1, 8, 2, 5376),                     # 320 shares, 352, 336
])
def test_divided_walks_against_whole_key_blocks(b, h, g, s):
    gen = torch.Generator(device=DEV).manual_seed(s + h)
    n = lambda *x: torch.randn(x, generator=gen, device=DEV)
    q, k, v, do, sinks = n(b, h, s, 64).bfloat16(), n(b, g, s, 64).bfloat16(), n(b, s, g, 64).bfloat16().transpose(1, 2), n(b, s, h, 64).bfloat16(), n(h)
    o, lse = ak.attention_forward(q, k, v, sinks, 0.125)
    got = ak.attention_backward(q, k, v, sinks, o, lse, do, 0.125)
    assert all(torch.equal(x, y) for x, y in zip(got, ak.attention_backward(q, k, v, sinks, o, lse, do, 0.125, split=True)))
    p = ak._base_params(q, k, v, sinks, None, 0.125, None, 0)
    want = torch.empty_like(q), torch.empty(k.shape, dtype=k.dtype, device=DEV), torch.empty(k.shape, dtype=k.dtype, device=DEV), torch.empty(h, device=DEV)
    p.o, p.lse, p.d_o = o.data_ptr(), lse.data_ptr(), do.data_ptr()
    p.dq, p.dk, p.dv, p.dsinks = (t.data_ptr() for t in want)
    for name, t, layout in (("o", o, "bshd"), ("do", do, "bshd"), ("dq", want[0], "bhsd"), ("dk", want[1], "bhsd"), ("dv", want[2], "bhsd")):
        ak._set(getattr(p, name + "_stride"), ak._strides_bhs(t, layout))
    _lib.call("gptoss_attn_bwd_static", p, torch.cuda.current_stream().cuda_stream)
    assert torch.equal(got[0], want[0]) and torch.equal(got[3], want[3])
    for name, x, y in (("dk", got[1].double(), want[1].double()), ("dv", got[2].double(), want[2].double())):
        # fp32 sums in another order: a value in a few thousand rounds to the other bf16 neighbour (2^-8 of it)
        assert (x - y).norm() <= 5e-4 * y.norm(), name
        assert bool(((x - y).abs() <= 2.0 ** -7 * y.abs() + 1e-4).all()), name
