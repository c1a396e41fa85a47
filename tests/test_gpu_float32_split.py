"""GPU tests of float32 attention on the bf16 matrix pipes (operands as three bf16 terms): edges of tiles, groups and parts, no further
from float64 than the fp32 matrix instruction, and the numbers the terms do not hold."""
import ctypes
import math

import pytest
import torch

from oracle import eager_ref as E
import test_gpu_float32 as TF
import test_gpu_parity as TP

pytestmark = pytest.mark.gpu
A = TF.A
SCALE, DEV = TF.SCALE, "cuda"


def _both(A, inp, window, seqlens=None, docs=None, start=0, backward=True):
    """(results, results of the fp32 matrix instruction)"""
    from oregon_gpt_oss_patching_amd import _lib
    from oregon_gpt_oss_patching_amd import attention_kernel as ak
    q, k, v, sinks, d_out = (t.to(DEV) for t in inp)
    lens = None if seqlens is None else torch.tensor(seqlens, dtype=torch.int32, device=DEV)
    ds = docs.to(DEV) if torch.is_tensor(docs) else None if docs is None else E.doc_start_from_lengths([docs] * q.shape[0], q.shape[2]).to(DEV).to(torch.int32)
    p = ak._base_params(q, k, v, sinks, lens, SCALE, window, start, ds)
    o, lse = A.attention_forward(q, k, v, sinks, SCALE, window, start, lens, ds)
    o2, lse2 = torch.empty_like(o), torch.empty_like(lse)
    p.o, p.lse = o2.data_ptr(), lse2.data_ptr()
    ak._set(p.o_stride, ak._strides_bhs(o2, "bshd"))
    assert _lib.load().gptoss_attn_split_bytes(ctypes.byref(p), int(backward)) > 0
    _lib.call("gptoss_attn_fwd", p, torch.cuda.current_stream().cuda_stream)
    if not backward:
        return (o, lse), (o2, lse2)
    args = (d_out, SCALE, window, 0, lens)
    return ((o, lse) + A.attention_backward(q, k, v, sinks, o, lse, *args, doc_start=ds),
            (o2, lse2) + A.attention_backward(q, k, v, sinks, o2, lse2, *args, doc_start=ds, split=True))


@pytest.mark.parametrize("b,h,g,s,w,lens,docs", [
    (1, 64, 8, 320, None, None, None),             # whole tiles, one key block of two and a half
    (1, 64, 8, 333, None, None, None),             # a last tile of 13 rows
    (2, 64, 8, 193, 128, None, None),              # one row past a tile, a window
    (3, 64, 8, 257, None, [257, 1, 130], None),    # padded rows, one of them a single token
    (1, 96, 8, 417, 33, None, None),               # twelve heads per KV head
    (2, 32, 8, 640, 500, None, None),              # four heads per KV head, a long window
    (1, 64, 8, 700, None, None, [5, 300, 32, 363]),
    (1, 8, 1, 2500, None, None, None),             # key blocks in parts of unequal number
])
def test_no_further_from_float64_than_the_fp32_instruction(A, b, h, g, s, w, lens, docs):
    print(f"case B={b} H={h} G={g} S={s} W={w} lens={lens} docs={docs}", flush=True)
    inp = list(E.make_inputs(7000 + s, b, h, g, s, 64, torch.float32))
    if lens:
        inp[4] = inp[4] * (torch.arange(s).view(1, s) < torch.tensor(lens).view(b, 1)).view(b, s, 1, 1)
    ds = E.doc_start_from_lengths([docs] * b, s) if docs else None
    new, old = _both(A, inp, w, lens, docs)
    f = [t.double().to(DEV) for t in inp]
    out, *grads = E.eager_attention_grads(*f, SCALE, w, 0, lens, ds)
    lse = E.logsumexp_rows(f[0], f[1], f[3], SCALE, w, 0, lens, ds)
    for name, x, y, ref in zip(("o", "lse", "dq", "dk", "dv", "dsinks"), new, old, (out, lse, *grads)):
        err, was = (float((t.double() - ref).norm() / ref.norm()) for t in (x, y))
        # dSinks is a cancelling sum over the rows: its error is the rows' common one, either way
        assert err <= min(2e-5, (float("inf") if name == "dsinks" else 1.05) * was), (name, err, was)
    again, _ = _both(A, inp, w, lens, docs)
    assert all(torch.equal(x, y) for x, y in zip(new, again))
    if lens:
        for i, n in enumerate(lens):
            for t in (new[0][i, n:], new[2][i, :, n:], new[3][i, :, n:], new[4][i, :, n:]):
                assert t.numel() == 0 or float(t.abs().max()) == 0.0


def _structured(kind, n):
    """Numbers whose terms do not average out."""
    g = torch.Generator().manual_seed(sum(n))
    if kind == "next to a bf16 number":                    # the first term leaves almost nothing, or almost all it can
        return torch.ldexp(torch.randn(n, generator=g).sign() * (1 + 2.0 ** -7 - 2.0 ** -23), torch.randint(-3, 2, n, generator=g))
    if kind == "1 to 1 + 2^-7":                            # dP - delta and the sums over the keys cancel
        return 1 + torch.rand(n, generator=g) * 2.0 ** -7
    if kind == "positive":
        return torch.rand(n, generator=g)
    out = torch.zeros(n)                                   # one product per contraction over head_dim at most
    return out.scatter(-1, torch.randint(0, n[-1], (*n[:-1], 1), generator=g), torch.randn((*n[:-1], 1), generator=g))


@pytest.mark.parametrize("b,h,g,s,w", [(1, 64, 8, 320, None), (1, 64, 8, 333, 33), (1, 32, 4, 700, 128)])
@pytest.mark.parametrize("kind", ["next to a bf16 number", "1 to 1 + 2^-7", "positive", "one number per row"])
def test_structured_operands(A, kind, b, h, g, s, w):
    print(f"case {kind} B={b} H={h} G={g} S={s} W={w}", flush=True)
    sinks = torch.randn(h, generator=torch.Generator().manual_seed(1))
    inp = [_structured(kind, n) for n in ((b, h, s, 64), (b, g, s, 64), (b, g, s, 64))] + [sinks, _structured(kind, (b, s, h, 64))]
    new, old = _both(A, inp, w)
    f = [t.double().to(DEV) for t in inp]
    out, *grads = E.eager_attention_grads(*f, SCALE, w)
    for name, x, y, ref in zip(("o", "lse", "dq", "dk", "dv"), new, old, (out, E.logsumexp_rows(f[0], f[1], f[3], SCALE, w), *grads)):
        err, was = (float((t.double() - ref).norm() / ref.norm()) for t in (x, y))
        # a sum of a few products: each is six additions to dK or dV here and one there, beside the errors of its P or dS (1.07 times)
        few = kind == "one number per row" and name in ("dk", "dv")
        assert err <= (1.12 if few else 1.05) * was, (name, err, was)


@pytest.mark.parametrize("sq,skv,w", [(256, 2049, None), (330, 1000, None), (330, 777, 100)])
def test_chunks_behind_a_cache(A, sq, skv, w):
    inp = E.make_inputs(7600 + sq, 1, 64, 8, sq, 64, torch.float32, skv=skv)
    new, old = _both(A, inp, w, start=skv - sq, backward=False)
    q, k, v, sinks, _ = (t.double().to(DEV) for t in inp)
    ref = E.eager_attention(q, k, v, sinks, SCALE, w, skv - sq)
    ref = ref[0] if isinstance(ref, tuple) else ref
    err, was = (float((t[0].double() - ref).norm() / ref.norm()) for t in (new, old))
    assert err <= min(2e-5, 1.05 * was), (err, was)
    assert float((new[1] - old[1]).abs().max()) <= 2e-5


@pytest.mark.parametrize("which,value", [("k", float("inf")), ("v", float("inf")), ("v", 1e30), ("v", float("nan")), ("q", 1e-35), ("q", 3e7),
                                         ("d_out", 1e-34), ("d_out", -float("inf")), ("v", 2.0 ** 24), ("v", 2.0 ** -100)])
def test_numbers_that_three_terms_do_not_hold(A, which, value):
    """One such number: what it reaches is what it reaches through the fp32 instruction."""
    inp = dict(zip(("q", "k", "v", "sinks", "d_out"), E.make_inputs(7700, 1, 64, 8, 333, 64, torch.float32)))
    t = inp[which]
    (t[0, 200, 5] if which == "d_out" else t[0, 2, 200])[7] = value
    new, old = _both(A, tuple(inp.values()), None)
    for name, x, y in zip(("o", "lse", "dq", "dk", "dv", "dsinks"), new, old):
        same = torch.isfinite(x) == torch.isfinite(y)
        assert bool(same.all()), (name, int((~same).sum()))
        assert torch.equal(torch.isnan(x), torch.isnan(y)), name
        ok = torch.isfinite(y)
        x, y = x[ok].double(), y[ok].double()
        assert float((x - y).norm()) <= 2e-5 * float(y.norm()), name


@pytest.mark.parametrize("b,s,w,lens,docs,row,at", [
    (2, 333, None, [150, 333], None, 0, 140),                  # the number in the last tile of a padded row
    (2, 333, None, [333, 150], None, 0, 200),
    (1, 700, None, None, [5, 300, 32, 363], 0, 200),           # in a document in the middle
    (1, 333, 100, None, None, 0, 200),                         # seen by a few tiles
    (1, 1056, None, None, None, 0, 900),                       # parts of 20 steps on eight heads: they start inside a pair of tiles
    (1, 2600, 500, None, None, 0, 64),
])
@pytest.mark.parametrize("which,value", [("k", float("inf")), ("v", 1e30), ("v", float("nan")), ("q", 1e-35), ("d_out", 1e-34), ("q", 3e7)])
def test_such_numbers_in_padded_packed_windowed_and_long_rows(A, which, value, b, s, w, lens, docs, row, at):
    """Row by row and column by column, so that a huge number hides nothing but itself."""
    print(f"case {which}={value} B={b} S={s} W={w} lens={lens} docs={docs}", flush=True)
    inp = dict(zip(("q", "k", "v", "sinks", "d_out"), E.make_inputs(7750 + s, b, 64, 8, s, 64, torch.float32)))
    t = inp[which]
    (t[row, at, 5] if which == "d_out" else t[row, 2, at])[7] = value
    if lens:
        inp["d_out"] = inp["d_out"] * (torch.arange(s).view(1, s) < torch.tensor(lens).view(b, 1)).view(b, s, 1, 1)
    _alike(*_both(A, tuple(inp.values()), w, lens, docs))


def _alike(new, old):
    for name, x, y in zip(("o", "lse", "dq", "dk", "dv"), new, old):
        assert torch.equal(torch.isfinite(x), torch.isfinite(y)) and torch.equal(torch.isnan(x), torch.isnan(y)), name
        ok = torch.isfinite(y)
        x, y = (torch.where(ok, t, 0.0).double() for t in (x, y))
        if name == "lse":
            assert bool(((x - y).abs() <= 2e-5 * (1 + y.abs())).all())
            continue
        # 2e-5 of the row's and of the column's size, as everywhere; a row that is much smaller than most (its products cancel): of those (which are not
        # the zeros of padding)
        rows, off = y.norm(dim=-1), (x - y).norm(dim=-1)
        most = rows[rows > 0].median()
        assert bool((off <= 2e-5 * (rows + most)).all()), (name, float((off / (rows + most)).max()))
        y, off = (t.reshape(-1, 64).norm(dim=0) for t in (y, x - y))
        assert bool((off <= 2e-5 * y).all()), (name, float((off / y).max()))


@pytest.mark.parametrize("sq,skv,w", [(330, 777, None), (256, 2049, None), (330, 777, 100)])
@pytest.mark.parametrize("which,value,at", [("k", float("inf"), 600), ("v", 1e30, 600), ("v", float("nan"), 40), ("q", 1e-35, 17)])
def test_such_numbers_behind_a_cache(A, which, value, at, sq, skv, w):
    inp = dict(zip(("q", "k", "v", "sinks", "d_out"), E.make_inputs(7760 + sq, 1, 64, 8, sq, 64, torch.float32, skv=skv)))
    inp[which][0, 2, at, 7] = value
    _alike(*_both(A, tuple(inp.values()), w, start=skv - sq, backward=False))


@pytest.mark.parametrize("which,value", [("v", float("inf")), ("v", -1e37), ("lse", -float("inf")), ("lse", float("inf"))])
def test_row_statistics_that_three_terms_do_not_hold(A, which, value):
    """A number that only the last row sees makes that row's delta infinite or large, or its lse is infinite: workgroups whose own operands are
    ordinary still get what the fp32 instruction gives."""
    q, k, v, sinks, d_out = (t.to(DEV) for t in E.make_inputs(7800, 1, 64, 8, 352, 64, torch.float32))
    for t in (q[0, :, -1], d_out[0, -1]):
        t.abs_()                                           # (what reaches dK has one sign: infinite or large, not NaN)
    if which == "v":
        v[0, 2, -1, 7] = value
    o, lse = A.attention_forward(q, k, v, sinks, SCALE)
    if which == "lse":
        lse[0, 5, -1] = value
    new, old = (A.attention_backward(q, k, v, sinks, o, lse, d_out, SCALE, split=split) for split in (False, True))
    if which == "v" and math.isfinite(value):              # (an infinite one is NaN times nothing in the rows that share its tile, either way)
        assert not torch.isnan(old[1][0, 2, :300]).any() and float(old[1][0, 2, :300].abs().min()) > 1e20
    for name, x, y in zip(("dq", "dk", "dv", "dsinks"), new, old):
        assert torch.equal(torch.isfinite(x), torch.isfinite(y)) and torch.equal(torch.isnan(x), torch.isnan(y)), name
        ok = torch.isfinite(y)
        assert bool(((x - y)[ok].abs() <= 1e-4 * y[ok].abs() + 2e-4).all()), name


@pytest.mark.parametrize("b,h,g,s,w,lens,docs", [
    (1, 64, 8, 5000, None, None, None),                        # four KV heads at a time
    (10, 64, 8, 1056, None, [1056, 700, 1, 0, 1055, 32, 33, 900, 1024, 1056], None),     # three KV heads of all rows at a time, then two
    (1, 28, 7, 15360, 500, None, None),                        # four KV heads, then three
    (3, 64, 8, 1700, None, None, [1, 932, 767]),               # four KV heads of all rows at a time
    (8, 16, 2, 5000, 500, [5000, 3, 4999, 0, 2500, 5000, 4000, 33], None),      # three batch rows at a time, then two
])
def test_some_rows_and_heads_at_a_time(A, b, h, g, s, w, lens, docs):
    """Calls whose records do not fit the scratch at once give what the fp32 instruction gives, and forward and dQ what each batch row gives by itself."""
    from oregon_gpt_oss_patching_amd import _lib
    from oregon_gpt_oss_patching_amd import attention_kernel as ak
    print(f"case B={b} H={h} G={g} S={s} W={w} lens={lens} docs={docs}", flush=True)
    inp = list(E.make_inputs(7900 + s, b, h, g, s, 64, torch.float32))
    p = ak._base_params(*(t.to(DEV) for t in inp[:4]), None, SCALE, w, 0, None)
    assert b * g * -(-s // 32) * (24576 + h // g * 24832) > _lib.load().gptoss_attn_split_bytes(ctypes.byref(p), 1) > 0
    new, old = _both(A, inp, w, lens, docs)
    for name, x, y in zip(("o", "lse", "dq", "dk", "dv"), new, old):
        # (each no further from float64 than 2e-5 of the result: 7e-7 at the most in test_no_further_from_float64_than_the_fp32_instruction)
        assert float((x - y).double().norm()) <= 2e-5 * float(y.double().norm()), name
    assert bool(((new[5] - old[5]).abs() <= 1e-4 * old[5].abs() + 1e-3).all())
    for i in range(b if b > 1 else 0):
        row = [t[i:i + 1] if t.dim() == 4 else t for t in inp]
        one, _ = _both(A, row, w, [lens[i]] if lens else None, docs)
        assert torch.equal(one[0], new[0][i:i + 1]) and torch.equal(one[1], new[1][i:i + 1]) and torch.equal(one[2], new[2][i:i + 1]), i


@pytest.mark.parametrize("sq,skv,w,start", [
    (330, 5000, 100, 4670), (330, 5000, 100, 131), (330, 5000, 100, 99), (330, 5000, 100, 1), (330, 5000, 100, 0),
    (321, 4100, 500, 3779),
    (320, 4099, 129, 2000),            # keys behind the last query
    (330, 600, 100, 500),              # queries behind the last key
    (330, 600, 100, 1200),             # none of them sees one
])
@pytest.mark.parametrize("on_device", [False, True])
def test_windows_behind_a_cache(A, sq, skv, w, start, on_device):
    """Records of the keys that some query sees, and of no others: the walks meet the right ones wherever the queries stand."""
    from oregon_gpt_oss_patching_amd import _lib
    from oregon_gpt_oss_patching_amd import attention_kernel as ak
    q, k, v, sinks, _ = (t.to(DEV) for t in E.make_inputs(7950 + start, 2, 32, 4, sq, 64, torch.float32, skv=skv))
    k[:, :, :max(0, start - w + 1)] = float("nan")             # (nobody sees them)
    at = torch.tensor([start], dtype=torch.int32, device=DEV) if on_device else None
    new = A.attention_forward(q, k, v, sinks, SCALE, w, 0 if on_device else start, q_offset_dev=at)
    p = ak._base_params(q, k, v, sinks, None, SCALE, w, start, None)
    o, lse = torch.empty_like(new[0]), torch.empty_like(new[1])
    p.o, p.lse = o.data_ptr(), lse.data_ptr()
    ak._set(p.o_stride, ak._strides_bhs(o, "bshd"))
    assert 0 < _lib.load().gptoss_attn_split_bytes(ctypes.byref(p), 0) <= 2 * 4 * (24576 + 4) * ((sq + w) // 32 + 2) + 256
    if start > w:
        k[:, :, :start - w + 1] = 0.0                          # (the other kernel multiplies what shares a tile, masked)
    _lib.call("gptoss_attn_fwd", p, torch.cuda.current_stream().cuda_stream)
    assert bool(torch.isfinite(o).all())
    # each no further from float64 than 2e-5 of the result (1.3e-6 at the most in test_chunks_behind_a_cache)
    assert float((new[0] - o).double().norm()) <= 2e-5 * float(o.double().norm())
    assert float((new[1] - lse).abs().max()) <= 2e-5


@pytest.mark.parametrize("b,h,g,s,w,lens,docs", [
    (1, 64, 8, 1030, None, None, [100] * 10 + [30]),
    (1, 64, 8, 700, None, None, [1] * 700),                    # every walk a single pair of tiles
    (1, 8, 1, 4100, None, None, [200] * 20 + [100]),           # many parts for few workgroups
    (1, 8, 1, 9000, None, None, [3, 1500, 1, 1, 40, 4000, 128, 127, 3200]),      # more key blocks than lanes
    (1, 8, 1, 4100, 500, None, [700, 1400, 2000]),
    (2, 64, 8, 1024, None, [100, 150], None),
    (9, 32, 4, 513, None, [513, 0, 1, 32, 33, 128, 129, 40, 200], None),         # one long row among short ones
    (3, 8, 1, 2500, None, [2500, 1200, 7], [900, 900, 700]),
    (1, 64, 8, 1030, None, None, "sliding"),                   # starts that move with the row
])
def test_walks_shortened_by_padding_and_documents(A, b, h, g, s, w, lens, docs):
    """dK / dV of key blocks whose walks are divided on the device: every step once, in slots that are there."""
    print(f"case B={b} H={h} G={g} S={s} W={w} lens={lens} docs={docs}", flush=True)
    if docs == "sliding":
        docs = (torch.arange(s) - 70).clamp(min=0).to(torch.int32).view(1, s).repeat(b, 1)
    inp = list(E.make_inputs(8000 + s, b, h, g, s, 64, torch.float32))
    if lens:
        inp[4] = inp[4] * (torch.arange(s).view(1, s) < torch.tensor(lens).view(b, 1)).view(b, s, 1, 1)
    new, old = _both(A, inp, w, lens, docs)
    _alike(new, old)
    again, _ = _both(A, inp, w, lens, docs)
    assert all(torch.equal(x, y) for x, y in zip(new, again))
