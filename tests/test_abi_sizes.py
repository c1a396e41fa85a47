"""Host-side tests of the sizing entry points: they answer before anything has been validated."""
import ctypes
import itertools

import pytest

from oregon_gpt_oss_patching_amd import _lib


def _params(dtype=0, b=1, h=64, g=8, sq=128, skv=128, window=0, **ptrs):
    p = _lib.new_params()
    p.dtype, p.B, p.H, p.G, p.Sq, p.Skv, p.D, p.window, p.scale = dtype, b, h, g, sq, skv, 64, window, 0.125
    for name, value in ptrs.items():
        setattr(p, name, value)
    return p


@pytest.mark.parametrize("h,g", [(4, 8), (1, 8), (6, 4), (0, 8), (8, 0), (-4, 8)])
def test_sizes_of_head_counts_that_the_calls_refuse(h, g):
    """Fewer query heads than KV heads (and other counts that do not divide): a size, whatever it is, and no division by zero."""
    lib = _lib.load()
    for dtype, sq, skv, window, doc in itertools.product((0, 1), (1, 64, 4096), (128, 4096), (0, 128), (None, 256)):
        p = _params(dtype, 1, h, g, sq, skv, window, doc_start=doc)
        assert lib.gptoss_attn_fwd_workspace_bytes(ctypes.byref(p)) == 0
        lib.gptoss_attn_workspace_bytes(ctypes.byref(p))
        assert lib.gptoss_attn_validate(ctypes.byref(p), 0) == -4


@pytest.mark.parametrize("sq,skv,window,start,shares", [
    (100, 8192, 128, 8092, 0),       # a window layer takes the window kernel, which cuts nothing
    (100, 8192, 0, 8092, 16),
    (100, 8192, 8192, 8092, 16),     # a window that reaches back past the first key is none
    (100, 8192, 8191, 8092, 0),
    (1024, 8192, 1024, 7168, 0),
])
def test_forward_scratch_follows_the_kernel_that_runs(sq, skv, window, start, shares):
    p = _params(sq=sq, skv=skv, window=window, q_offset=start)
    rows = 64 * sq
    assert _lib.load().gptoss_attn_fwd_workspace_bytes(ctypes.byref(p)) == shares * rows * (64 + 2) * 4
    if window > skv - 1:             # (where the position is on the device, the host does not know that)
        p.q_offset_dev = 256
        assert _lib.load().gptoss_attn_fwd_workspace_bytes(ctypes.byref(p)) == 0
