"""Builds a C++ check of the library's host/device functions for the CPU (the HIP compiler's host
half only) and runs it."""
import os
import shutil
import subprocess

import pytest

from conftest import PKG_DIR, ROOT


def run_check(name, tmp_path, sanitize=False):
    hipcc = next((c for c in ("/opt/rocm/bin/hipcc", shutil.which("hipcc")) if c and os.path.exists(c)), None)
    if hipcc is None:
        pytest.skip("hipcc not found")
    exe = str(tmp_path / name)
    cmd = [hipcc, "--cuda-host-only", "-x", "hip", "-std=c++17", "-O1", "-Wno-unused-value",
           "-I", os.path.join(PKG_DIR, "csrc"), os.path.join(ROOT, "tests", name + ".cpp"), "-o", exe]
    if sanitize:
        cmd += ["-Xarch_host", "-fsanitize=address,undefined", "-g"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-4000:]
    res = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, (res.stdout + res.stderr)[-4000:]
    return res.stdout
