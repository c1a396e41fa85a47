"""Tracing the operators without a GPU: sizes that are symbols stay symbols (shape-only tensors that say they are on a GPU)."""
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.symbolic_shapes import DimDynamic, ShapeEnv, StatelessSymbolicContext

import oregon_gpt_oss_patching_amd as A


def _symbols():
    """A batch and a length that are symbols, 3 and 100 where a number is asked for."""
    env = ShapeEnv()
    mode = FakeTensorMode(shape_env=env)
    ctx = StatelessSymbolicContext(dynamic_sizes=[DimDynamic.DYNAMIC, DimDynamic.DYNAMIC])
    return env, mode, mode.from_tensor(torch.empty((3, 100), device="meta"), symbolic_context=ctx, static_shapes=False).shape


def _tensors(b, s):
    q = torch.empty((b, 64, s, 64), dtype=torch.bfloat16, device="cuda")
    k = torch.empty((b, 8, s, 64), dtype=torch.bfloat16, device="cuda")
    v = torch.empty((b, s, 8, 64), dtype=torch.bfloat16, device="cuda").transpose(1, 2)
    return q, k, v, torch.empty((64,), dtype=torch.bfloat16, device="cuda")


def _untied(env):
    return not env.replacements and not [g for g in env.guards if "Eq" in str(g.expr)]


def test_batch_and_length_stay_symbols():
    for window in (None, 128):
        for padded in (False, True):
            env, mode, (b, s) = _symbols()
            with mode, torch.no_grad():
                lens = torch.empty((b,), dtype=torch.int32, device="cuda") if padded else None
                out = A.attention(*_tensors(b, s), 0.125, window, None, lens)
            assert tuple(map(str, out.shape)) == (str(b), str(s), "64", "64") and _untied(env)


def test_query_offset_stays_a_symbol():
    """(a decoding loop whose position is a Python integer: one program for all positions)"""
    env, mode, (b, s) = _symbols()
    with mode, torch.no_grad():
        torch.ops.gptoss_attn.attention(*_tensors(b, s), 0.125, 0, 7 * s, None, None)
    assert _untied(env)


def test_documents_of_packed_rows_stay_symbols():
    env, mode, (b, s) = _symbols()
    with mode:
        out = A.doc_start_from_position_ids(torch.empty((b, s), dtype=torch.int64, device="cuda"))
    assert tuple(map(str, out.shape)) == (str(b), str(s)) and out.dtype == torch.int32 and _untied(env)
