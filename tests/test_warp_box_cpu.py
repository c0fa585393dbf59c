"""The pieces of source rows that a warp loads: inside the batch buffer wherever they are loaded without a look at its ends."""
import os
import shutil
import subprocess

import pytest

from test_dma_waitcnt_cpu import ROOT


def test_unchecked_pieces_lie_in_the_buffer(tmp_path):
    if not shutil.which("g++") or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("needs g++ and the HIP headers")
    exe = str(tmp_path / "warp_box")
    fma = ["-mfma", "-mavx2"] if " fma " in open("/proc/cpuinfo").read() else []
    subprocess.run(["g++", "-O2", "-std=c++17", "-w", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", *fma,
                    "-I" + os.path.join(ROOT, "rocal_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "warp_box.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
