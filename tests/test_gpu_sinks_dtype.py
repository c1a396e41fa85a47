"""GPU tests of the sink logits and their gradient in bfloat16: the bits of the calls with the same logits widened to
float32, and the float32 gradient rounded once, on every route that reads or writes them."""
import pytest
import torch

from oracle import eager_ref as E

pytestmark = pytest.mark.gpu
SCALE, DEV = 0.125, "cuda"


@pytest.mark.parametrize("dtype,b,h,g,s,skv,window,start", [
    (torch.bfloat16, 1, 8, 2, 200, 200, 0, 0),        # sliced dK/dV: the gradient comes out of the launch that adds the slices
    (torch.bfloat16, 1, 6, 2, 33, 33, 0, 0),          # a single slice: a launch of its own
    (torch.bfloat16, 2, 8, 2, 130, 130, 128, 0),      # sliding window, one pass
    (torch.bfloat16, 1, 8, 2, 130, 130, 200, 0),      # a window that covers the row: full causal
    (torch.bfloat16, 1, 8, 1, 160, 160, 64, 0),       # one-pass window forward
    (torch.bfloat16, 1, 64, 8, 1, 700, 0, 699),       # decoding, cut over the keys
    (torch.bfloat16, 1, 8, 2, 2, 40, 0, 38),          # decoding, uncut
    (torch.float32, 1, 8, 2, 600, 600, 0, 0),         # float32 tensors with bfloat16 logits, sliced
    (torch.float32, 1, 4, 2, 40, 40, 32, 0),
])
def test_bf16_sinks_give_the_bits_of_widened_ones(dtype, b, h, g, s, skv, window, start):
    import oregon_gpt_oss_patching_amd as A
    A.attention_kernel  # noqa: B018 (registers the operators)
    print(f"case {dtype} B={b} H={h} G={g} S={s} Skv={skv} W={window} start={start}", flush=True)
    q, k, v, sinks, d_out = (t.to(DEV) for t in E.make_inputs(5000 + s, b, h, g, s, 64, dtype, skv=skv))
    bf = sinks.to(torch.bfloat16)
    ops = torch.ops.gptoss_attn
    o, lse = ops.fwd(q, k, v, bf.float(), SCALE, window, start, None, None)
    o2, lse2 = ops.fwd(q, k, v, bf, SCALE, window, start, None, None)
    assert torch.equal(o, o2) and torch.equal(lse, lse2)
    wide = ops.bwd(q, k, v, bf.float(), o, lse, d_out, SCALE, window, start, None, None, True)
    got = ops.bwd(q, k, v, bf, o, lse, d_out, SCALE, window, start, None, None, True)
    own = ops.bwd(q, k, v, bf, o, lse, d_out, SCALE, window, start, None, None, True, None, True)
    for w, x, y in zip(wide, got, own):
        assert torch.equal(w, x) and torch.equal(w.to(y.dtype), y)
    assert got[3].dtype == torch.float32 and own[3].dtype == torch.bfloat16
