"""Generated code of the resize kernels for rows at any byte phase, of the nearest-pixel kernel and of the one whose tiles are dealt: as for the streaming bilinear
kernel, a wait for a window's loads that leaves N operations outstanding needs N stores in the held-back group behind them."""
import os
import re

import pytest

from test_dma_waitcnt_cpu import HIPCC, _device_assembly


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
@pytest.mark.parametrize("src,name,instances", [("rmx_kernels_resize_fast.hip", "rmx_resize_fast_kernel", 30), ("rmx_kernels_resize_near.hip", "rmx_resize_near_kernel", 12),
                                                ("rmx_kernels_resize_split.hip", "rmx_resize_split_kernel", 42)])
def test_held_back_stores_cover_the_wait_count(src, name, instances):
    text = _device_assembly(src)
    checked = 0
    for f in re.split(r"\n(?=_ZN3rmx\d+%s[^\n]*:\s)" % name, text):
        m = re.match(r"(_ZN3rmx\d+%s\S*):" % name, f)
        if not m:
            continue
        body = f.split("s_endpgm")[0]
        n = max([int(x) for x in re.findall(r"^\s*s_waitcnt vmcnt\((\d+)\)\s*$", body, re.M)], default=0)
        lines = body.splitlines()
        loads = [i for i, l in enumerate(lines) if "global_load_lds" in l]
        assert loads and "scratch_" not in body, m.group(1)
        held = next((b for b in re.split(r"\n(?=\.LBB\d+_\d+:)", "\n".join(lines[loads[-1] + 1:])) if re.search(r"^\s*global_store", b, re.M)), "")
        if n:
            assert len(re.findall(r"^\s*global_store", held, re.M)) >= n and "global_load_lds" not in held, m.group(1)
        checked += 1
    assert checked == instances
