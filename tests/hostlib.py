"""Compiles a snippet that includes the kernels' own headers for the host, so
that the CPU tests evaluate the rules and formulas that the kernels use."""
from __future__ import annotations

import ctypes
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def host_lib(tmp_path, code: str) -> ctypes.CDLL:
    src, so = str(tmp_path / "snippet.hip"), str(tmp_path / "snippet.so")
    with open(src, "w") as f:
        f.write(code)
    subprocess.run([HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "hcgrid_amd", "csrc"),
                    src, "-o", so], check=True)
    return ctypes.CDLL(so)
