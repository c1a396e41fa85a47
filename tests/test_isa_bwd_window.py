"""Checks on the compiled code of attn_bwd_window_kernel (hipcc cross-compiles without a GPU).

Twelve wavefronts, three per SIMD, leave 168 registers per lane.  The walk needs all of them: what the compiler spills beside must stay out of the loops (one
register, stored and loaded again in front of and behind them), and the scalar values that it parks in vector registers out of the steps' own.
"""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    hipcc = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    from oregon_gpt_oss_patching_amd import build as B
    d = tmp_path_factory.mktemp("isa_bwd_window")
    src, out = d / "unit.hip", d / "unit.s"
    src.write_text(f'#include "{os.path.join(ROOT, "oregon_gpt_oss_patching_amd", "csrc", "attn_bwd_window.h")}"\n')
    flags = [f for f in B.HIPCC_FLAGS if f not in ("-fPIC", "-shared")]
    proc = subprocess.run([hipcc, *flags, "-S", "--cuda-device-only", "-o", str(out), str(src)], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-2000:]
    return out.read_text()


def test_three_wavefronts_per_simd(assembly):
    kernel = re.search(r"\.amdhsa_kernel _ZN6gptoss22attn_bwd_window_kernel(.*?)\.end_amdhsa_kernel", assembly, re.S).group(1)
    n = {x: int(y) for x, y in re.findall(r"\.amdhsa_(private_segment_fixed_size|next_free_vgpr)\s+(\d+)", kernel)}
    assert n["next_free_vgpr"] <= 168
    assert n["private_segment_fixed_size"] <= 8


def test_no_spills_in_the_loops(assembly):
    code = re.search(r"\n_ZN6gptoss22attn_bwd_window_kernel\w*:(.*?)\.Lfunc_end", assembly, re.S).group(1).split("\n")
    label = {line.split(":")[0]: i for i, line in enumerate(code) if line.startswith(".LBB")}
    loops = []
    for i, line in enumerate(code):
        m = re.match(r"\ts_c?branch\w*\s+(\.LBB\w+)", line)
        if m and label[m.group(1)] < i:
            loops.append(code[label[m.group(1)]:i + 1])
    assert not any("scratch_" in line for loop in loops for line in loop)
    # the steps of the owners (16 MFMAs) and of the helpers (20): the shortest loop around each
    for mfmas in (16, 20):
        steps = [loop for loop in loops if sum("v_mfma" in line for line in loop) == mfmas]
        assert steps, mfmas
        assert sum("v_readlane" in line for line in min(steps, key=len)) <= 4
