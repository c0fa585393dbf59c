"""The host side of the library on a HIP runtime made of host memory (tests/cpp/host_runtime.cpp): what calls that succeed and fail
leave behind, without a GPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++") or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("needs g++ and the HIP headers")
    exe = str(tmp_path_factory.mktemp("host_runtime") / "host_runtime")
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "rocal_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "host_runtime.cpp"), "-o", exe, "-ldl"], check=True)
    return exe


@pytest.mark.parametrize("what", ["ring", "failed upload", "failed launch"])
def test_host_side(program, what):
    from rocal_amd import _lib
    r = subprocess.run([program, _lib.LIB_PATH, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
