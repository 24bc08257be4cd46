"""Host-only check of the reconstruction core's arguments
(candmc_amd/csrc/hr_kernel.hip) in tests/cxx/test_hr_args.cpp: refused before
anything is launched.  Compiled with hipcc as host code against the built
library; no GPU call is made."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"
LIB = os.path.join(ROOT, "candmc_amd", "libcandmc_qr.so")


@pytest.mark.skipif(not os.path.exists(HIPCC) or not os.path.exists(LIB),
                    reason="needs hipcc and the built library")
def test_outputs_of_the_inverse_need_it(tmp_path):
    exe = str(tmp_path / "hr_args")
    cmd = [HIPCC, "-O1", "-std=c++17", "-I" + os.path.join(ROOT, "include"),
           "-I" + os.path.join(ROOT, "candmc_amd", "csrc"),
           os.path.join(ROOT, "tests", "cxx", "test_hr_args.cpp"),
           "-L" + os.path.dirname(LIB), "-lcandmc_qr", "-Wl,-rpath," + os.path.dirname(LIB), "-o", exe]
    subprocess.run(cmd, check=True, capture_output=True, timeout=600)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stdout + run.stderr
    assert "hr args ok" in run.stdout
