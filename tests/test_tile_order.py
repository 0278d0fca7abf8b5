"""Order of the uniform tree's tile lists (csrc/tree.cpp heaviest_first), on the host."""
import os
import subprocess

import pytest

from conftest import REPO

CSRC = os.path.join(REPO, "spectral-bslpm_amd", "csrc")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("tiles") / "tile_order_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I",
                           os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"), "-I", CSRC,
                           os.path.join(CSRC, "tree.cpp"),
                           os.path.join(REPO, "tests", "cpp", "tile_order_check.cpp"), "-o", out])
    return out


# one level (no interactions between panels of two levels), short lists with one and two tiles per
# panel, and lists either side of the limit (2,556, then 8,190 tiles)
@pytest.mark.parametrize("levels,degree,leaf_degree,theta", [(1, 4, 4, 0.7), (3, 6, 6, 0.7), (4, 8, 7, 0.7),
                                                             (4, 10, 10, 0.5), (5, 8, 5, 0.7), (6, 6, 6, 0.7)])
def test_tile_order(exe, levels, degree, leaf_degree, theta):
    out = subprocess.run([exe, str(levels), str(degree), str(leaf_degree), str(theta)], capture_output=True, text=True)
    assert out.returncode == 0, (out.returncode, out.stdout, out.stderr)
