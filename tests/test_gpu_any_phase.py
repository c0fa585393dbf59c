"""Bilinear and nearest resizes from source rows at any byte phase, bit for bit against the oracle: row strides of every remainder
mod 4, images packed at every byte address, windows on both edges and on the last byte of the buffer, destinations of 1 to 9 pixels,
rows whose last x-tile is a few pixels wide (narrow tiles forced by a small LDS budget), mirrored, every format."""
import numpy as np
import pytest

from oracle import orc
from rocal_amd import ops, workloads as wl

pytestmark = pytest.mark.gpu
COMBOS = [(ops.NCHW, ops.FP16), (ops.NCHW, ops.FP32), (ops.NCHW, ops.UINT8), (ops.NHWC, ops.FP16), (ops.NHWC, ops.FP32), (ops.NHWC, ops.UINT8)]


@pytest.mark.parametrize("layout,dtype", COMBOS)
@pytest.mark.parametrize("interp", [ops.LINEAR, ops.NEAREST])
@pytest.mark.parametrize("W", [149, 150, 151, 152])
@pytest.mark.parametrize("packed", [False, True])
def test_rows_at_every_phase(ctx, ctx_undealt, ctx_dma_small, ctx_dma_split, layout, dtype, interp, W, packed):
    import torch
    rng = np.random.default_rng(W * 100 + 10 * layout + dtype + (7 if packed else 0))
    n, H, OH, OW = 12, 90, 70, 140
    img = rng.integers(0, 256, (n, H, W, 3), dtype=np.uint8)
    widths, heights = np.full(n, W, np.uint32), np.full(n, H, np.uint32)
    if packed:
        widths, heights = rng.integers(100, W + 1, n).astype(np.uint32), rng.integers(60, H + 1, n).astype(np.uint32)
    roi = np.empty((n, 4), np.uint32)
    for i in range(n):
        iw, ih = int(widths[i]), int(heights[i])
        w, h = int(rng.integers(20, iw + 1)), int(rng.integers(20, ih + 1))
        roi[i] = (int(rng.integers(0, iw - w + 1)), int(rng.integers(0, ih - h + 1)), w, h)
    roi[0] = (0, 0, widths[0], heights[0])
    roi[n - 1] = (widths[-1] - 30, heights[-1] - 20, 30, 20)  # ends on the last byte of the buffer
    roi[1] = (3, 5, 1, 1)
    dw = rng.integers(40, OW + 1, n).astype(np.uint32)
    dh = rng.integers(10, OH + 1, n).astype(np.uint32)
    dw[2:11] = np.arange(1, 10)          # destinations of 1 .. 9 pixels from windows of 20 and fewer per pixel
    roi[2:11, 2] = np.minimum(roi[2:11, 2], 3 * dw[2:11])
    dw[0], dw[11] = 133, 67              # 128 + 5 and 64 + 3: a last tile of fewer than 8 columns where tiles are narrow
    mirror = rng.integers(0, 2, n).astype(np.uint32)
    norm = dtype != ops.UINT8
    scale, bias = orc.cmn_scale_bias(wl.MEAN, wl.STD, n)
    quant = norm and interp == ops.LINEAR
    exp = orc.resize(img, roi, dw, dh, OH, OW, interp=interp, mirror=mirror, scale=scale if norm else None, bias=bias if norm else None, layout=layout,
                     dtype=dtype, flags=orc.F_QUANTIZE_U8 if quant else 0)
    if packed:
        sizes = widths.astype(np.int64) * heights * 3
        offsets = np.cumsum(sizes) - sizes
        flat = torch.from_numpy(np.concatenate([img[i, :heights[i], :widths[i]].reshape(-1) for i in range(n)])).cuda()
    src = flat if packed else torch.from_numpy(img).cuda()
    for c in (ctx, ctx_undealt, ctx_dma_small, ctx_dma_split):
        op = ops.Resize(c, ops.desc(n, H, W, ops.NHWC, ops.UINT8), ops.desc(n, OH, OW, layout, dtype), interp, flags=ops.F_QUANTIZE_U8 if quant else 0)
        if packed:
            op.set_ragged_source(offsets.astype(np.uint64), widths, heights, flat.numel())
        if norm:
            op.update_cmn(roi, dw, dh, scale, bias, mirror)
        else:
            op.update(roi, dw, dh, mirror)
        want = {ops.NEAREST: "rmx_resize_near_kernel", ops.LINEAR: "rmx_resize_fast_kernel" if packed or W % 4 else "rmx_resize_dma_kernel"}[interp]
        dealt = "split=" in op.plan
        assert not dealt or c in (ctx, ctx_dma_split), op.plan
        # (a window too tall for the small budget takes the general kernel)
        assert op.kernel_name == ("rmx_resize_split_kernel" if dealt else want) or c in (ctx_dma_small, ctx_dma_split), op.plan
        out = op.alloc_output(fill=5)
        op.launch(src, out)
        c.sync()
        got = out.cpu().numpy()
        keep = np.full_like(exp, 5)
        for i in range(n):
            x = (i, slice(None), slice(0, dh[i]), slice(0, dw[i])) if layout == ops.NCHW else (i, slice(0, dh[i]), slice(0, dw[i]))
            keep[x] = exp[x]
        assert np.array_equal(got.view(np.uint8), keep.view(np.uint8)), (op.plan, [i for i in range(n) if not np.array_equal(got[i], keep[i])])
