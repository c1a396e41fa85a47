"""The checks of test_isa_fwd_pipe on the compiled code of attn_fwd_pipe_kernel's packed-document instantiation."""
import pytest

import test_isa_fwd_pipe as T
from test_isa_fwd_pipe import test_every_micro_slot_of_the_loop_has_its_mfma, test_loop_has_no_scratch_access_and_no_compiler_made_vmcnt_wait  # noqa: F401


@pytest.fixture(scope="module")
def kernel_lines(tmp_path_factory):
    import os
    import re
    import subprocess
    hipcc = T._hipcc()
    if hipcc is None:
        pytest.skip("hipcc not found")
    from oregon_gpt_oss_patching_amd import build as B
    d = tmp_path_factory.mktemp("isa_fwd_documents")
    src, out = d / "unit.hip", d / "unit.s"
    src.write_text('#include "%s"\ntemplate __global__ void gptoss::attn_fwd_pipe_kernel<true, true>(const gptoss::KArgs);\n'
                   % os.path.join(T.CSRC, "attn_fwd_pipe.h"))
    flags = [f for f in B.HIPCC_FLAGS if f not in ("-fPIC", "-shared")]
    proc = subprocess.run([hipcc, *flags, "-S", "--cuda-device-only", "-o", str(out), str(src)], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-2000:]
    m = re.search(r"^(_ZN6gptoss\d+%s\w*):[^\n]*\n(.*?)\.end_amdhsa_kernel" % T.KERNEL, out.read_text(), re.S | re.M)
    assert m, "kernel not found in the assembly"
    return m.group(2).split("\n")
