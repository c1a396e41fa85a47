"""GPU tests of how the full-causal kernels divide their work: rows packed from documents whose ends lie on, before and
behind tile and key-block edges (the dK/dV walk ends with the document), key blocks cut into slices, and right-padded
batches whose rows are dealt to the workgroups in rotation.  Against the eager oracle."""
import pytest
import torch

from oracle import eager_ref as E
import test_gpu_parity as TP

pytestmark = pytest.mark.gpu
A = TP.A
SCALE = TP.SCALE


@pytest.mark.parametrize("b,h,g,docs", [
    (1, 8, 2, [64, 128, 256, 64]),                      # documents of whole tiles
    (1, 8, 2, [63, 129, 1, 255, 65, 2]),                # one off every edge, one-token documents
    (1, 16, 2, [1, 700]),
    (1, 8, 1, [300, 1, 1, 1, 900, 97]),
    (2, 8, 4, [511, 513, 200]),
    (1, 8, 2, [2048, 70, 1990]),                        # 4108 tokens: three rounds of the search for a document's end
])
@pytest.mark.parametrize("w", [None, 128])
def test_packed_rows_vs_eager_oracle(A, b, h, g, docs, w):
    print(f"case B={b} H={h} G={g} docs={docs} W={w}", flush=True)
    s = sum(docs)
    inp = E.make_inputs(5000 + s, b, h, g, s, 64, torch.bfloat16)
    ds = E.doc_start_from_lengths([docs] * b, s)
    TP.compare_all(TP.run_hip(A, *inp, w, 0, None, ds), TP.oracle_eager(*inp, w, 0, None, ds))


@pytest.mark.parametrize("b,h,g,s,lens", [
    (2, 8, 1, 383, None),               # six slices of one query tile
    (3, 4, 2, 130, None),               # three query tiles of two heads: no slice below eight steps
    (4, 8, 1, 448, [448, 1, 65, 300]),  # slices of a padded batch, rows in rotation
    (5, 8, 2, 257, [257, 256, 255, 64, 7]),
])
def test_sliced_and_rotated_batches_vs_eager_oracle(A, b, h, g, s, lens):
    print(f"case B={b} H={h} G={g} S={s} lens={lens}", flush=True)
    inp = E.make_inputs(5100 + s, b, h, g, s, 64, torch.bfloat16)
    if lens:
        inp = inp[:4] + (TP.mask_dout(inp[4], lens),)
    TP.compare_all(TP.run_hip(A, *inp, None, 0, lens), TP.oracle_eager(*inp, None, 0, lens))


@pytest.mark.parametrize("b,h,g,sq,skv,start,lens", [
    (1, 8, 2, 64, 64, 0, None),             # one tile
    (1, 8, 2, 65, 65, 0, None),             # a last tile of one row and one key
    (2, 16, 4, 127, 127, 0, None),
    (1, 8, 2, 300, 1000, 700, None),        # an offset inside a tile: the diagonal lies across two tiles
    (1, 8, 2, 129, 449, 320, None),         # ... on a tile boundary, with a last tile of one key
    (1, 8, 2, 200, 1000, 300, None),        # a cache longer than what the queries see
    (1, 4, 1, 100, 90, 10, None),           # fewer keys than positions
    (3, 8, 2, 333, 333, 0, [333, 64, 1]),   # padded rows of a ragged batch
    (2, 8, 2, 100, 600, 500, [600, 520]),   # padded rows behind an offset: queries past the row's length
])
@pytest.mark.parametrize("lift", [0.0, 40.0])
def test_full_causal_forward_of_any_length_vs_eager_oracle(A, b, h, g, sq, skv, start, lens, lift):
    """The pipelined forward off whole tiles.  lift: the second half of the keys is scaled so that a row's later logits stand
    far above its first tile's (the frozen softmax reference is found too low and the workgroup repeats its walk)."""
    print(f"case B={b} H={h} G={g} Sq={sq} Skv={skv} start={start} lens={lens} lift={lift}", flush=True)
    q, k, v, sinks, _ = E.make_inputs(5200 + sq + skv, b, h, g, sq, 64, torch.bfloat16, skv=skv)
    if lift:
        k[:, :, skv // 2:] *= lift
    args = (SCALE, None, start, lens)
    o, lse = A.attention_forward(*(t.to("cuda") for t in (q, k, v, sinks)), *args)
    f = [t.float() for t in (q, k, v, sinks)]
    TP.check("o", o, E.eager_attention(*f, *args))
    ref = E.logsumexp_rows(f[0], f[1], f[3], *args).float()
    assert float((lse.cpu() - ref).abs().max()) <= TP.LSE_TOL * (1 if not lift else 1 + float(ref.abs().max()) / 64)   # (fp32 logits of order 300)
    if lens:
        for i, n in enumerate(lens):
            assert (o[i, max(n - start, 0):] == 0).all()


@pytest.mark.parametrize("docs", [[100, 28, 200], [1, 63, 64, 65, 190], [300, 10, 10, 10, 500], [129, 700]])
def test_packed_forward_with_sharply_peaked_rows(A, docs):
    """Documents that end inside a workgroup's rows, logits of order 40: the rows that start afresh at the diagonal tile take a
    softmax reference of their own."""
    s = sum(docs)
    print(f"case docs={docs}", flush=True)
    q, k, v, sinks, _ = E.make_inputs(5300 + s, 2, 8, 2, s, 64, torch.bfloat16)
    q, k = q * 3, k * 3
    ds = E.doc_start_from_lengths([docs] * 2, s)
    o, lse = A.attention_forward(*(t.to("cuda") for t in (q, k, v, sinks)), SCALE, None, doc_start=ds)
    f = [t.float() for t in (q, k, v, sinks)]
    TP.check("o", o, E.eager_attention(*f, SCALE, None, 0, None, ds))
    assert float((lse.cpu() - E.logsumexp_rows(f[0], f[1], f[3], SCALE, None, 0, None, ds).float()).abs().max()) <= TP.LSE_TOL


@pytest.mark.parametrize("b,h,g,s,lens,docs", [
    (1, 16, 2, 2049, None, None),                    # a query tile of one row on top of the walk, cut into slices
    (1, 8, 1, 2303, [2303], None),                   # ... of 63 rows; a single KV head
    (3, 8, 2, 2111, [2111, 2048, 700], None),        # padded rows that end below the tile that sticks out, and in it
    (33, 8, 8, 449, None, None),                     # more than 512 key blocks: whole blocks
    (1, 16, 2, 2100, None, [64, 192, 1, 63, 257, 700, 823]),    # documents inside wavefronts, on their edges, across workgroups
    (1, 8, 2, 2048, None, [2048]),
    (2, 8, 2, 2300, None, [1, 2299]),
    (1, 8, 2, 2500, None, [5] * 500),                # many documents in one wavefront's keys
    (2, 8, 2, 2200, [2200, 1500], [900, 700, 600]),  # packed and padded
])
def test_64_key_backward_of_any_length_vs_eager_oracle(A, b, h, g, s, lens, docs):
    """attn_bwd_dkdv64_kernel off whole tiles and with packed documents, every gradient, and the same bits on a second run."""
    print(f"case B={b} H={h} G={g} S={s} lens={lens} docs={docs}", flush=True)
    inp = E.make_inputs(5400 + s + b, b, h, g, s, 64, torch.bfloat16)
    if lens:
        inp = inp[:4] + (TP.mask_dout(inp[4], lens),)
    ds = E.doc_start_from_lengths([docs] * b, s) if docs else None
    got = TP.run_hip(A, *inp, None, 0, lens, ds)
    o, lse, dq, dk, dv, dsinks = (t.detach().cpu() for t in got)
    rds = torch.zeros(h, dtype=torch.float64)
    for i in range(b):
        one = [t[i:i + 1] for t in inp[:3]] + [inp[3], inp[4][i:i + 1]]
        ro, rlse, rdq, rdk, rdv, rds_i = TP.oracle_eager(*one, None, 0, [lens[i]] if lens else None, ds[i:i + 1] if docs else None)
        # Documents of five tokens: a dK element is scale * sum of dS q over 5 rows x 4 heads, with |dS| up to p (1 - p) |dP - delta| ~
        # 4 (dP is a sum of 64 products of N(0, 1) values) and |q| ~ 2, so rounding dS to bf16 (2^-9 relative) moves it by up to
        # 2^-9 * 20 * 4 * 2 / 8 = 4e-2; everywhere else the bound of 2e-2 holds.
        atol = 4e-2 if docs and max(docs) <= 5 else 2e-2
        for name, x, y in (("o", o, ro), ("dq", dq, rdq), ("dk", dk, rdk), ("dv", dv, rdv)):
            TP.check(name, x[i:i + 1], y, atol=atol)
        assert float((lse[i:i + 1] - rlse.float()).abs().max()) <= TP.LSE_TOL
        rds += rds_i.double()
    TP.check("dsinks", dsinks, rds.float(), atol=None)
    again = TP.run_hip(A, *inp, None, 0, lens, ds)
    assert all(torch.equal(x, y) for x, y in zip(got, again))


@pytest.mark.parametrize("b,h,g,s,lens", [
    (2, 8, 4, 64 * 5 + 1, None),                    # a last chunk of less than two tiles
    (1, 16, 8, 64 * 97, None),                      # 97 tiles x 8 heads: chunks of four on 256 compute units, a last one of a single tile
    (3, 16, 8, 1999, [1999, 700, 65]),              # chunks of three
])
def test_window_backward_chunks_vs_eager_oracle(A, b, h, g, s, lens):
    """The single-pass window backward where the chunk length follows the rounds of workgroups."""
    print(f"case B={b} H={h} G={g} S={s} lens={lens}", flush=True)
    inp = E.make_inputs(5500 + s, b, h, g, s, 64, torch.bfloat16)
    if lens:
        inp = inp[:4] + (TP.mask_dout(inp[4], lens),)
    TP.compare_all(TP.run_hip(A, *inp, 128, 0, lens), TP.oracle_tiled(*inp, 128, 0, lens))
