"""The streaming triangular kernels, that with eight accumulator sets (columns 64 apart) at the vertical ratios where a sample changes from all
eight sets to the lower four (1/2), at the windows' ends, and with so few output rows that every row has a set of its own; rows in the kernel's
arguments and in a table, in strips of every length. Bit for bit against the oracle and the ring kernel."""
import numpy as np
import pytest

from oracle import orc
from rocal_amd import ops, workloads as wl

pytestmark = pytest.mark.gpu


def _run(c, img, roi, rs, crop, out_hw, layout, dtype, mirror):
    import torch
    n, H, W = img.shape[:3]
    op = ops.Resize(c, ops.desc(n, H, W, ops.NHWC, ops.UINT8), ops.desc(n, out_hw[0], out_hw[1], layout, dtype), ops.TRIANGULAR)
    s, b = orc.cmn_scale_bias(wl.MEAN, wl.STD, n)
    op.update_cmn(roi, rs[:, 0].copy(), rs[:, 1].copy(), s, b, mirror, crop_roi=crop)
    out = op.alloc_output(fill=5)
    op.launch(torch.from_numpy(img).cuda(), out)
    c.sync()
    return op, out.cpu().numpy()


@pytest.mark.parametrize("layout,dtype", [(ops.NCHW, ops.FP16), (ops.NHWC, ops.FP32)])
@pytest.mark.parametrize("rows,compact", [(0, 1), (4, 1), (9, 1), (23, 0)])
@pytest.mark.parametrize("adjacent", [0, 1])
def test_ratios_around_one_half_and_short_windows(layout, dtype, rows, compact, adjacent):
    from conftest import _ctx_with_env
    rng = np.random.default_rng(70 + rows)
    OH, OW = 96, 64
    # source rows, resized rows: ratios just below, at and just above 1/2, below 1/3, between, 1, above 1; 3 to 9 output rows
    heights = [(47, 96), (48, 96), (49, 96), (27, 96), (32, 96), (61, 96), (95, 96), (96, 96), (97, 96), (150, 96), (2, 4), (2, 3), (3, 8), (4, 9), (40, 81), (41, 82)]
    n, H, W = len(heights), 152, 80
    img = wl.smooth_noise(rng, n, H, W, sigma=1.0)
    roi = np.array([[i % 5, (0, H - h)[i & 1], 60 + i % 3, h] for i, (h, _) in enumerate(heights)], np.uint32)  # at the source's first or last rows
    rs = np.array([[OW - i % 9, r] for i, (_, r) in enumerate(heights)], np.uint32)
    if compact:  # one resized size, so that the rows travel in the arguments
        rs[:] = (OW - 2, 96)
        roi[:, 3] = np.maximum(roi[:, 3], 27)
        roi[:, 1] = [(0, H - int(h))[i & 1] for i, h in enumerate(roi[:, 3])]
    mirror = (np.arange(n) % 3 == 0).astype(np.uint32)
    # the whole resized image, and a crop of it (its first and last written rows are not the window's)
    crop = np.stack([np.full(n, 2), rs[:, 1] // 5, rs[:, 0] - 7, rs[:, 1] - rs[:, 1] // 5 - rs[:, 1] // 6], 1).astype(np.uint32)
    c = _ctx_with_env(RMX_TUNE_TRI_ROWS=rows, RMX_TUNE_COMPACT=compact, RMX_TUNE_TRI_ADJ=adjacent)
    ring = _ctx_with_env(RMX_TUNE_TRI_RING=1)
    s, b = orc.cmn_scale_bias(wl.MEAN, wl.STD, n)
    try:
        for cr in (None, crop):
            op, got = _run(c, img, roi, rs, cr, (OH, OW), layout, dtype, mirror)
            kernel, form = ("rmx_resize_tri_adj_kernel", "adjacent=1") if adjacent else ("rmx_resize_tri_dma_kernel", "rows_in_flight=8")
            assert op.kernel_name == kernel and form in op.plan and ("rows=arguments" if compact else "rows=table") in op.plan, op.plan
            _, other = _run(ring, img, roi, rs, cr, (OH, OW), layout, dtype, mirror)
            assert np.array_equal(got.view(np.uint8), other.view(np.uint8)), op.plan
            if cr is None:
                exp = orc.resize(img, roi, rs[:, 0], rs[:, 1], OH, OW, interp=orc.TRIANGULAR, mirror=mirror, scale=s, bias=b, layout=layout, dtype=dtype)
                for i, (w, h) in enumerate(rs):
                    g, e = (got[i, :, :h, :w], exp[i, :, :h, :w]) if layout == ops.NCHW else (got[i, :h, :w], exp[i, :h, :w])
                    assert np.array_equal(np.ascontiguousarray(g).view(np.uint8), np.ascontiguousarray(e).view(np.uint8)), "sample %d (%s)" % (i, op.plan)
    finally:
        c.close()
        ring.close()
