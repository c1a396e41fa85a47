"""GPU tests of the forward for a few queries on a key / value cache (attn_decode_kernel): against the eager oracle at the
edges of its tiles, slices and (query, head) blocks, with windows, padded rows, caches that are longer than what is filled
and offsets read on the device."""
import pytest
import torch

from oracle import eager_ref as E

pytestmark = pytest.mark.gpu
SCALE, DEV = 0.125, "cuda"


@pytest.fixture(scope="module")
def A():
    import oregon_gpt_oss_patching_amd as A_
    from oregon_gpt_oss_patching_amd import _lib
    _lib.load()
    return A_


@pytest.mark.parametrize("b,h,g,sq,skv,start,w,lens", [
    (1, 64, 8, 1, 2049, 2048, None, None),         # slices of one tile per wavefront, a last tile of one key
    (3, 16, 2, 1, 1000, 999, None, None),
    (1, 8, 8, 1, 33, 32, None, None),              # one slice: the kernel writes the results itself
    (1, 64, 8, 1, 1, 0, None, None),               # a single key
    (2, 8, 1, 4, 700, 696, None, None),            # 32 pairs: the last of one column block
    (2, 8, 1, 5, 700, 695, None, None),            # 40 pairs: two column blocks
    (1, 64, 1, 1, 517, 516, None, None),           # 64 query heads of one KV head
    (1, 6, 2, 7, 300, 293, None, None),            # a group of three heads
    (1, 64, 8, 1, 4096, 4095, 128, None),          # sliding window at the end of a long cache
    (2, 8, 2, 3, 640, 300, 100, None),             # the queries stand in the middle of the cache
    (2, 8, 2, 2, 640, 126, None, None),
    (3, 8, 2, 2, 900, 700, None, [900, 701, 5]),   # padded rows: whole, a dead second query, dead altogether
    (1, 8, 2, 8, 8, 0, None, None),                # self-attention of eight tokens
    (1, 8, 1, 1, 1024, 1023, None, None),          # the most keys one workgroup walks alone, and one more
    (1, 8, 1, 1, 1025, 1024, None, None),
    (1, 8, 1, 1, 257, 256, None, None),            # nine tiles of eight wavefronts, the last of one key
    (1, 8, 1, 8, 640, 632, None, None),            # 64 pairs, unsliced and sliced
    (1, 8, 1, 8, 641, 633, None, None),
    (130, 8, 4, 1, 300, 299, None, None),          # 520 KV heads: four wavefronts, unsliced
    (4, 8, 1, 1, 40000, 39999, 128, None),         # a window at the end of a long cache, unsliced
])
@pytest.mark.parametrize("on_device", [False, True])
def test_decode_vs_eager_oracle(A, b, h, g, sq, skv, start, w, lens, on_device):
    print(f"case B={b} H={h} G={g} Sq={sq} Skv={skv} start={start} W={w} lens={lens} on_device={on_device}", flush=True)
    q, k, v, sinks, _ = E.make_inputs(4000 + skv + sq, b, h, g, sq, 64, torch.bfloat16, skv=skv)
    off = torch.tensor([start], dtype=torch.int32, device=DEV) if on_device else None
    args = (sinks.to(DEV), SCALE, w, 0 if on_device else start, lens)
    o, lse = A.attention_forward(q.to(DEV), k.to(DEV), v.to(DEV), *args, q_offset_dev=off)
    f = [t.float() for t in (q, k, v, sinks)]
    ref = E.eager_attention(*f, SCALE, w, start, lens)
    ref_lse = E.logsumexp_rows(f[0], f[1], f[3], SCALE, w, start, lens)
    # the bf16 path's bounds: 1e-2 relative (2-norm), 2e-2 absolute plus half an ulp of the bf16 result, lse 1e-3
    o = o.float().cpu()
    assert torch.isfinite(o).all()
    assert float((o.double() - ref.double()).norm()) <= 1e-2 * float(ref.double().norm())
    assert bool(((o - ref).abs() <= 2e-2 + 2.0 ** -8 * ref.abs()).all())
    assert float((lse.cpu() - ref_lse.float()).abs().max()) <= 1e-3
    again, lse2 = A.attention_forward(q.to(DEV), k.to(DEV), v.to(DEV), *args, q_offset_dev=off)
    assert torch.equal(again.float().cpu(), o) and torch.equal(lse, lse2)


def test_decode_without_scratch_and_under_graph_replay(A):
    """delta == NULL runs the same kernel uncut; a captured call gives the eager result on every replay."""
    from oregon_gpt_oss_patching_amd import _lib
    from oregon_gpt_oss_patching_amd import attention_kernel as ak
    q, k, v, sinks, _ = (t.to(DEV) for t in E.make_inputs(4100, 2, 16, 2, 1, 64, torch.bfloat16, skv=1500))
    s32 = sinks.float().contiguous()
    o, lse = A.attention_forward(q, k, v, sinks, SCALE, None, 1499)
    o1, lse1 = torch.full_like(o, float("nan")), torch.full_like(lse, float("nan"))
    p = ak._base_params(q, k, v, s32, None, SCALE, None, 1499)
    p.o, p.lse = o1.data_ptr(), lse1.data_ptr()
    ak._set(p.o_stride, ak._strides_bhs(o1, "bshd"))
    _lib.call("gptoss_attn_fwd", p, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert float((o1.float() - o.float()).abs().max()) <= 2.0 ** -7 and float((lse1 - lse).abs().max()) <= 1e-5
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        A.attention_forward(q, k, v, s32, SCALE, None, 1499)
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        og, lg = A.attention_forward(q, k, v, s32, SCALE, None, 1499)
    for _ in range(3):
        og.zero_()
        k.add_(0.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(og, o) and torch.equal(lg, lse)


@pytest.mark.parametrize("b,sq,skv,start,lens", [(1, 8, 129, 121, None), (1, 1, 2049, 2048, None), (2, 3, 600, 597, [600, 40])])
def test_decode_without_sink(A, b, sq, skv, start, lens):
    """Sink logits of -inf: the plain softmax, also for rows that see nothing of some slice's or wavefront's keys."""
    print(f"case B={b} Sq={sq} Skv={skv} start={start} lens={lens}", flush=True)
    q, k, v, sinks, _ = E.make_inputs(4200 + skv, b, 8, 1, sq, 64, torch.bfloat16, skv=skv)
    none = torch.full_like(sinks, float("-inf"))
    o, _ = A.attention_forward(q.to(DEV), k.to(DEV), v.to(DEV), none.to(DEV), SCALE, None, start, lens)
    ref = E.eager_attention(q.float(), k.float(), v.float(), torch.full_like(sinks.float(), -1e4), SCALE, None, start, lens)
    o = o.float().cpu()
    live = torch.ones(b, sq, dtype=torch.bool) if lens is None else torch.arange(start, start + sq)[None] < torch.tensor(lens)[:, None]
    # the bf16 path's bound, as above
    assert bool(((o - ref).abs() <= 2e-2 + 2.0 ** -8 * ref.abs())[live].all())
