"""Generated code of the streaming triangular kernel: its tables of vertical coefficients are written and read by the wavefront
itself, so no access to them waits for memory. The loads of the next source rows are in flight while a row is filtered, and a
wait for the vector memory counter in front of an LDS access (which the compiler adds where it takes the access for one of the
loads' own) would end that."""
import os
import re

import pytest

from test_dma_waitcnt_cpu import HIPCC, _device_assembly


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
@pytest.mark.parametrize("unit", ["2", "4", "8_nchw", "8_nhwc"])
def test_tables_of_vertical_coefficients_wait_for_no_load(unit):
    text = _device_assembly("rmx_kernels_tri_dma_%s.hip" % unit)
    names = 0
    for f in re.split(r"\n(?=_ZN3rmx25rmx_resize_tri_dma_kernel[^\n]*:\s)", text):
        m = re.match(r"(_ZN3rmx25rmx_resize_tri_dma_kernel\S*):", f)
        if not m:
            continue
        names += 1
        ins = [l.strip() for l in f.split("s_endpgm")[0].splitlines() if l.startswith("\t") and not l.strip().startswith(".")]
        # (instructions in #ASMSTART .. #ASMEND are the source's own; comments start with ";")
        own = False
        for k, line in enumerate(ins):
            own = own or "#ASMSTART" in line
            if "#ASMEND" in line:
                own = False
            if own or not (line.startswith("s_waitcnt") and "vmcnt" in line):
                continue
            after = next((i for i in ins[k + 1:] if not i.startswith(";")), "")
            assert not re.match(r"ds_(read|write)(2)?_b(64|128)", after), "%s: %s in front of %s" % (m.group(1), line, after)
    assert names
