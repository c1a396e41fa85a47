"""GPU tests of the pipelined forward with its keys cut into shares (few queries on a long cache): at the edges of tiles and shares,
shares that no row of a block sees, offsets on the device, padded rows, sharply rising logits, against the eager oracle."""
import pytest
import torch

from oracle import eager_ref as E
import test_gpu_parity as TP

pytestmark = pytest.mark.gpu
A = TP.A
SCALE, DEV = TP.SCALE, "cuda"


@pytest.mark.parametrize("b,h,g,sq,skv,start,lens", [
    (1, 8, 1, 17, 1536, 1519, None),              # three shares of eight tiles
    (1, 8, 1, 64, 1600, 1536, None),
    (1, 8, 2, 65, 1601, 1536, None),              # a last tile of one key, a last query block of one row
    (1, 4, 1, 130, 8200, 8070, None),             # sixteen shares
    (1, 8, 1, 100, 2000, 0, None),                # the queries stand at the start of the cache: two tiles for all shares
    (1, 8, 2, 100, 2000, 700, None),
    (1, 8, 1, 100, 2000, 1950, None),             # fewer keys than positions
    (3, 8, 2, 40, 1700, 1600, [1700, 1610, 90]),  # padded rows: whole, cut inside the queries, dead altogether
])
@pytest.mark.parametrize("lift", [0.0, 40.0])
@pytest.mark.parametrize("on_device", [False, True])
def test_shares_vs_eager_oracle(A, b, h, g, sq, skv, start, lens, lift, on_device):
    """lift: the second half of the keys is scaled, so that the shares' references lie far apart and a frozen one is found too low."""
    print(f"case B={b} H={h} G={g} Sq={sq} Skv={skv} start={start} lens={lens} lift={lift} on_device={on_device}", flush=True)
    q, k, v, sinks, _ = E.make_inputs(7000 + sq + skv, b, h, g, sq, 64, torch.bfloat16, skv=skv)
    if lift:
        k[:, :, skv // 2:] *= lift
    vd = v.transpose(1, 2).contiguous().to(DEV).transpose(1, 2)
    off = torch.tensor([start], dtype=torch.int32, device=DEV) if on_device else None
    args = (q.to(DEV), k.to(DEV), vd, sinks.to(DEV), SCALE, None, 0 if on_device else start, lens, None, off)
    o, lse = A.attention_forward(*args)
    f = [t.float() for t in (q, k, v, sinks)]
    TP.check("o", o, E.eager_attention(*f, SCALE, None, start, lens))
    ref = E.logsumexp_rows(f[0], f[1], f[3], SCALE, None, start, lens).float()
    assert float((lse.cpu() - ref).abs().max()) <= TP.LSE_TOL * (1 if not lift else 1 + float(ref.abs().max()) / 64)   # (fp32 logits of order 300)
    again, lse2 = A.attention_forward(*args)
    assert torch.equal(again, o) and torch.equal(lse2, lse)


def test_shares_without_sink_without_scratch_and_under_graph_replay(A):
    from oregon_gpt_oss_patching_amd import _lib
    from oregon_gpt_oss_patching_amd import attention_kernel as ak
    q, k, v, sinks, _ = (t.to(DEV) for t in E.make_inputs(7100, 1, 8, 1, 100, 64, torch.bfloat16, skv=2500))
    none = torch.full_like(sinks, float("-inf"))
    o, _ = A.attention_forward(q, k, v, none, SCALE, None, 2400)
    f = [t.float().cpu() for t in (q, k, v)]
    TP.check("o", o, E.eager_attention(*f, torch.full((8,), -1e4), SCALE, None, 2400))
    s32 = sinks.float().contiguous()
    o, lse = A.attention_forward(q, k, v, s32, SCALE, None, 2400)
    # delta == NULL: the same call uncut
    o1, lse1 = torch.full_like(o, float("nan")), torch.full_like(lse, float("nan"))
    p = ak._base_params(q, k, v, s32, None, SCALE, None, 2400)
    p.o, p.lse = o1.data_ptr(), lse1.data_ptr()
    ak._set(p.o_stride, ak._strides_bhs(o1, "bshd"))
    assert _lib.load().gptoss_attn_fwd_workspace_bytes(p) <= _lib.load().gptoss_attn_workspace_bytes(p)
    _lib.call("gptoss_attn_fwd", p, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert float((o1.float() - o.float()).abs().max()) <= 2.0 ** -6 and float((lse1 - lse).abs().max()) <= 1e-5
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        A.attention_forward(q, k, v, s32, SCALE, None, 2400)
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        og, lg = A.attention_forward(q, k, v, s32, SCALE, None, 2400)
    for _ in range(3):
        og.zero_()
        k.add_(0.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(og, o) and torch.equal(lg, lse)
