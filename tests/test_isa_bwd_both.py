"""Checks on the compiled code of attn_bwd_both_kernel (hipcc cross-compiles without a GPU): its route counts on two workgroups per compute unit, a dQ and a dK/dV
one among them, which share the kernel's LDS array rather than having one each, and at most half of the registers.
"""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_two_workgroups_per_compute_unit(tmp_path):
    hipcc = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    from oregon_gpt_oss_patching_amd import build as B
    src, out = tmp_path / "unit.hip", tmp_path / "unit.s"
    forms = ("false, false", "false, true", "true, false")
    src.write_text(f'#include "{os.path.join(ROOT, "oregon_gpt_oss_patching_amd", "csrc", "attn_bwd.h")}"\n' +
                   "".join(f"template __global__ void gptoss::attn_bwd_both_kernel<{f}>(const gptoss::KArgs, int, int);\n" for f in forms))
    flags = [f for f in B.HIPCC_FLAGS if f not in ("-fPIC", "-shared")]
    proc = subprocess.run([hipcc, *flags, "-S", "--cuda-device-only", "-o", str(out), str(src)], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-2000:]
    kernels = re.findall(r"\.amdhsa_kernel _ZN6gptoss20attn_bwd_both_kernel(.*?)\.end_amdhsa_kernel", out.read_text(), re.S)
    assert len(kernels) == len(forms)
    for k in kernels:
        n = {x: int(y) for x, y in re.findall(r"\.amdhsa_(group_segment_fixed_size|private_segment_fixed_size|next_free_vgpr)\s+(\d+)", k)}
        assert n["group_segment_fixed_size"] <= 160 * 1024 // 2
        assert n["private_segment_fixed_size"] == 0
        assert n["next_free_vgpr"] <= 256                      # four wavefronts of each workgroup on four SIMDs of 512
