"""GPU test of the document starts formed from position ids, against the tensor operations a CPU tensor takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,docs", [(1, [1]), (3, [7, 1, 1, 300]), (1, [1023, 1, 1]), (2, [1024, 1024]), (1, [5000, 3, 70]),
                                    (2, [1025, 2046, 1, 1024]), (1, [1] * 3000)])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
def test_document_starts_match_the_cpu(b, docs, dtype):
    from oregon_gpt_oss_patching_amd import doc_start_from_position_ids as f
    print(f"case B={b} docs={docs[:8]} dtype={dtype}", flush=True)
    s = sum(docs)
    g = torch.Generator().manual_seed(s)
    rows = []
    for i in range(b):
        order = [docs[j] for j in torch.randperm(len(docs), generator=g).tolist()]
        rows.append(torch.cat([torch.arange(n) + (5 * i) % 7 for n in order]))     # restarts at 0, 5, 3: any step but + 1 is a start
    pos = torch.stack(rows).to(dtype)
    want = f(pos)
    for view in (pos.cuda(), pos.cuda().t().contiguous().t(), pos[:1].cuda().expand(b, s)):
        got = f(view)
        assert got.dtype == torch.int32 and got.is_contiguous() and got.shape == (b, s)
        assert torch.equal(got.cpu(), want if view.stride(0) or b == 1 else want[:1].expand(b, s))
    jumps = torch.randint(0, 4, (b, s), generator=g).cumsum(1).to(dtype)             # positions that go on by 0 .. 3
    assert torch.equal(f(jumps.cuda()).cpu(), f(jumps))
