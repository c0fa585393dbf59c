"""Generated code of the streaming triangular kernel: its tables of vertical coefficients are written and read by the wavefront
itself, so no access to them waits for memory. The loads of the next source rows are in flight while a row is filtered, and a
wait for the vector memory counter in front of an LDS access (which the compiler adds where it takes the access for one of the
loads' own), however far in front, would end that."""
import os
import re

import pytest

from test_dma_waitcnt_cpu import HIPCC, _device_assembly


def _idle_waits(body):
    """The compiler's own waits for the vector memory counter that wait for no load into registers: only loads into LDS and stores are
    outstanding then, and what stands behind the wait does not need them. (Operations complete in order: a wait for n leaves the n
    youngest outstanding. Instructions in #ASMSTART .. #ASMEND are the source's own, its waits are meant.)"""
    own, flight, idle = False, [], []
    for line in body.splitlines():
        line = line.strip()
        if "#ASMSTART" in line or "#ASMEND" in line:
            own = "#ASMSTART" in line
        elif re.match(r"(global|buffer|flat|scratch)_", line):
            flight.append(bool(re.match(r"(global|buffer|flat|scratch)_load_(?!lds)", line)) and not line.endswith(" lds"))
        elif re.match(r"s_waitcnt .*vmcnt\(", line):
            n = int(re.search(r"vmcnt\((\d+)\)", line).group(1))
            done, flight = flight[:max(0, len(flight) - n)], flight[max(0, len(flight) - n):]
            if not own and not any(done):
                idle.append(line)
    return idle


def test_idle_waits_are_told_from_needed_ones():
    load, into_lds = "\tglobal_load_dword v1, v2, s[0:1]\n", "\tglobal_load_lds_dwordx4 v2, s[0:1]\n"
    table = "\tv_add_u32_e32 v3, 16, v3\n\tds_read_b128 v[4:7], v3\n"
    assert _idle_waits(into_lds + "\ts_waitcnt vmcnt(0)\n" + table) == ["s_waitcnt vmcnt(0)"]
    assert _idle_waits(load + into_lds + "\ts_waitcnt vmcnt(1)\n" + table) == []
    assert _idle_waits(load + into_lds + "\ts_waitcnt vmcnt(1)\n\ts_waitcnt vmcnt(0) lgkmcnt(0)\n" + table) == ["s_waitcnt vmcnt(0) lgkmcnt(0)"]
    assert _idle_waits(into_lds + "\t;;#ASMSTART\n\ts_waitcnt vmcnt(0)\n\t;;#ASMEND\n" + table) == []


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
        assert not _idle_waits(f.split(".Lfunc_end")[0]), m.group(1)
    assert names


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
@pytest.mark.parametrize("unit", ["nchw", "nhwc", "nchw_any", "nhwc_any"])
def test_kernel_of_neighbouring_columns_counts_its_stores(unit):
    """rmx_resize_tri_adj_kernel waits for its loads into LDS with s_waitcnt vmcnt(0 | NS | 2 NS | 4 NS), NS the fewest store instructions that an
    output row can become: three planes, or one interleaved run. The compiler makes the stores, so every place that stores a row must
    hold as many, nothing may spill to scratch memory, and the numbered waits are the source's own. Its tables of vertical
    coefficients wait for no load; one idle wait stands on the path of rows that the lanes store at the buffer's end."""
    text = _device_assembly("rmx_kernels_tri_adj_%s.hip" % unit)
    ns = 3 if unit.startswith("nchw") else 1
    checked = 0
    for f in re.split(r"\n(?=_ZN3rmx25rmx_resize_tri_adj_kernel[^\n]*:\s)", text):
        m = re.match(r"(_ZN3rmx25rmx_resize_tri_adj_kernel\S*):", f)
        if not m:
            continue
        body = f.split(".Lfunc_end")[0]
        assert not re.search(r"^\s*(scratch_|buffer_|flat_)", body, re.M), m.group(1)
        own = [int(x) for part in re.findall(r"#ASMSTART(.*?)#ASMEND", body, re.S) for x in re.findall(r"s_waitcnt vmcnt\((\d+)\)", part)]
        assert set(own) == {0, ns, 2 * ns, 4 * ns}, "%s: waits %s" % (m.group(1), sorted(set(own)))
        places = 0
        for block in re.split(r"\n(?=\.LBB\d+_\d+:|; %bb\.\d+:)", body):
            stores = re.findall(r"^\s*global_store_\w+", block, re.M)
            assert not stores or len(stores) >= ns, "%s: a row in %d stores" % (m.group(1), len(stores))
            places += bool(stores)
        assert places >= 6 * 2  # six numbers of taps, samples that shrink and that grow
        assert "global_load_lds_dwordx4" in body
        assert len(_idle_waits(body)) <= 1, m.group(1)
        checked += 1
    assert checked == 9
