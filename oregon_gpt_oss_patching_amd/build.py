"""Compiles the HIP attention library for gfx950 with hipcc (no torch headers), and the PyTorch operators over it.

`python -m oregon_gpt_oss_patching_amd.build` or `build_library()` and `build_torch_ops()`; the results,
libgptoss_attn.so and libgptoss_torch.so, are placed beside this file and loaded by `_lib.py`.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sysconfig

_HERE = os.path.dirname(os.path.abspath(__file__))
SOURCE = os.path.join(_HERE, "csrc", "gptoss_attn.hip")
LIBRARY = os.path.join(_HERE, "libgptoss_attn.so")
TORCH_SOURCE = os.path.join(_HERE, "csrc", "torch_ops.cpp")
TORCH_LIBRARY = os.path.join(_HERE, "libgptoss_torch.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    # packed fp32 VALU ops are kept off for every kernel in this library
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # MFMA results stay in ordinary vector registers unless a kernel pins an accumulator to the AGPR half
    # itself (the 64-key dK/dV kernel does, through inline assembly)
    "-mllvm", "-amdgpu-mfma-vgpr-form",
]


def hipcc_path() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found; set HIPCC or install ROCm")


def _run(cmd, verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd))
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"{os.path.basename(cmd[0])} failed:\n{proc.stdout}\n{proc.stderr}")


def build_library(verbose: bool = False) -> str:
    _run([hipcc_path(), *HIPCC_FLAGS, "-o", LIBRARY, SOURCE], verbose)
    return LIBRARY


def build_torch_ops(verbose: bool = False) -> str:
    """The operators link to libgptoss_attn.so beside them; build that one first."""
    import torch
    root = os.path.dirname(torch.__file__)
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(hipcc_path())))
    _run([shutil.which("g++") or "c++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
          "-isystem", os.path.join(root, "include"), "-isystem", os.path.join(root, "include", "torch", "csrc", "api", "include"),
          "-isystem", os.path.join(rocm, "include"), "-isystem", sysconfig.get_paths()["include"], "-o", TORCH_LIBRARY, TORCH_SOURCE,
          "-L" + os.path.join(root, "lib"), "-lc10", "-ltorch_cpu", "-lc10_hip", "-ltorch_hip", "-L" + _HERE, "-lgptoss_attn", "-Wl,-rpath,$ORIGIN"], verbose)
    return TORCH_LIBRARY


if __name__ == "__main__":
    print(build_library(verbose=True))
    print(build_torch_ops(verbose=True))
