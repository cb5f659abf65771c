"""Errors of kernel launches (launch.hpp), with the runtime replaced by one that refuses them: no GPU takes part."""
import os
import shutil
import subprocess

import pytest

from tests.cpp.build import ROOT

ROCM = "/opt/rocm/include"


@pytest.mark.skipif(not os.path.exists(os.path.join(ROCM, "hip", "hip_runtime.h")) or shutil.which("g++") is None, reason="needs g++ and HIP's headers")
def test_errors_are_reported_once(tmp_path):
    exe = str(tmp_path / "launch_error_check")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I", ROCM, "-I", os.path.join(ROOT, "rmlx_amd", "csrc"),
                           "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "cpp", "launch_error_check.cpp"), "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=30)
    assert r.returncode == 0 and "launch errors ok" in r.stdout, r.stdout + r.stderr
