"""The ratios of a resize from the sizes in its records: the same as the host's divisions, and made without a division."""
import os
import re
import shutil
import subprocess

import pytest

from test_dma_waitcnt_cpu import HIPCC, ROOT, _device_assembly


def test_ratio_is_the_quotient(tmp_path):
    if not shutil.which("g++") or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("needs g++ and the HIP headers")
    exe = str(tmp_path / "quotients")
    fma = ["-mfma", "-mavx2"] if " fma " in open("/proc/cpuinfo").read() else []
    subprocess.run(["g++", "-O3", "-std=c++17", "-w", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", *fma,
                    "-I" + os.path.join(ROOT, "rocal_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "quotients.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
@pytest.mark.parametrize("src,name", [("rmx_kernels_resize_dma.hip", "rmx_resize_dma_kernel"), ("rmx_kernels_resize_fast.hip", "rmx_resize_fast_kernel"),
                                      ("rmx_kernels_resize_fast.hip", "rmx_resize_runs_kernel"), ("rmx_kernels_resize_near.hip", "rmx_resize_near_kernel")])
def test_no_division_in_front_of_the_first_load(src, name):
    """Every wavefront runs its kernel's beginning in front of its first source load: no division there."""
    found = 0
    for f in re.split(r"\n(?=_ZN3rmx\d+%s[^\n]*:\s)" % name, _device_assembly(src)):
        m = re.match(r"(_ZN3rmx\d+%s\S*):" % name, f)
        if not m:
            continue
        found += 1
        assert "v_div_" not in f.split("s_endpgm")[0].split("global_load_lds")[0], m.group(1)
    assert found >= 5
