"""The copies between host and device memory, on the CPU: tests/host_stage_check.cpp with stand-ins for the HIP calls."""
import os
import shutil
import subprocess

import pytest

from tests.conftest import ROOT

ROCM_INCLUDE = "/opt/rocm/include"


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(ROCM_INCLUDE), reason="needs g++ and HIP's headers")
def test_host_stage(tmp_path):
    exe = str(tmp_path / "host_stage_check")
    cmd = ["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM_INCLUDE}",
           os.path.join(ROOT, "tests", "host_stage_check.cpp"), "-o", exe, "-pthread"]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "0 failed checks" in r.stdout, (r.stdout + r.stderr)[-4000:]
