"""Check on the compiled code of attn_f32_dkdv_kernel (hipcc cross-compiles without a GPU): it shares its body with the walk over pairs of tiles of
attn_f32_split.h and must not pay for that one's index arithmetic (2505 instructions; 2763 with both walks in one).
"""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_key_blocks_walk_has_its_own_indexing(tmp_path):
    hipcc = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    from oregon_gpt_oss_patching_amd import build as B
    src, out = tmp_path / "unit.hip", tmp_path / "unit.s"
    csrc = os.path.join(ROOT, "oregon_gpt_oss_patching_amd", "csrc")
    src.write_text("".join(f'#include "{os.path.join(csrc, name)}"\n' for name in ("attn_bwd.h", "attn_f32.h")))
    flags = [f for f in B.HIPCC_FLAGS if f not in ("-fPIC", "-shared")]
    proc = subprocess.run([hipcc, *flags, "-S", "--cuda-device-only", "-o", str(out), str(src)], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-2000:]
    code = re.search(r"\n_ZN6gptoss20attn_f32_dkdv_kernel\w*:(.*?)\.Lfunc_end", out.read_text(), re.S).group(1)
    assert len(re.findall(r"^\t[a-z]\w+", code, re.M)) <= 2630
