"""log_wide (csrc/fasttab.hpp), the table logarithm of the FP64 log pair kernels, against the
long-double logarithm on the host."""
import os
import subprocess

from conftest import REPO


def test_wide_log_accuracy(tmp_path):
    exe = str(tmp_path / "wide_log_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-DSBSLPM_HD=", "-I",
                           os.path.join(REPO, "spectral-bslpm_amd", "csrc"),
                           os.path.join(REPO, "tests", "cpp", "wide_log_check.cpp"), "-o", exe])
    out = subprocess.run([exe], capture_output=True, text=True)
    print(out.stdout)
    assert out.returncode == 0, out.stdout + out.stderr
