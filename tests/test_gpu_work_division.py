"""GPU tests of how the full-causal kernels divide their work: rows packed from documents whose ends lie on, before and
behind tile and key-block edges (the dK/dV walk ends with the document), key blocks cut into slices, and right-padded
batches whose rows are dealt to the workgroups in rotation.  Against the eager oracle."""
import pytest
import torch

from oracle import eager_ref as E
import test_gpu_parity as TP

pytestmark = pytest.mark.gpu
A = TP.A


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
