"""Rows per tile (csrc/tree.hpp), which decide between a row per lane and lane copies, on the host."""
import os
import subprocess

from conftest import REPO

CSRC = os.path.join(REPO, "spectral-bslpm_amd", "csrc")


def test_tile_rows(tmp_path):
    exe = str(tmp_path / "tile_rows_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I",
                           os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"), "-I", CSRC,
                           os.path.join(CSRC, "tree.cpp"), os.path.join(CSRC, "irreg_tree.cpp"),
                           os.path.join(REPO, "tests", "cpp", "tile_rows_check.cpp"), "-o", exe])
    out = subprocess.run([exe], capture_output=True, text=True)
    print(out.stdout)
    assert out.returncode == 0, (out.returncode, out.stdout, out.stderr)
