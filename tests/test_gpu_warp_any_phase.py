"""Warps from source rows at any byte phase: row strides of every remainder mod 4, padded and packed at every byte address, windows
on both edges and on the last byte of the buffer, images a few pixels wide, maps that enlarge, shrink (wide LDS rows, gathers from
memory) and point outside, destinations of 1 to 9 pixels and of odd widths. Bytes against the oracle; every format bit for bit
against the same images in a batch whose rows are multiples of 4 bytes."""
import numpy as np
import pytest

from oracle import orc
from rocal_amd import ops

pytestmark = pytest.mark.gpu
COMBOS = [(ops.NHWC, ops.UINT8), (ops.NCHW, ops.UINT8), (ops.NCHW, ops.FP16), (ops.NHWC, ops.FP16), (ops.NCHW, ops.FP32), (ops.NHWC, ops.FP32)]


def _batch(W, H, n, rng):
    widths, heights = rng.integers(max(1, W - 40), W + 1, n).astype(np.uint32), rng.integers(max(1, H - 30), H + 1, n).astype(np.uint32)
    roi, affine = np.empty((n, 4), np.uint32), np.empty((n, 6), np.float32)
    for i in range(n):
        iw, ih = int(widths[i]), int(heights[i])
        w, h = int(rng.integers(1, iw + 1)), int(rng.integers(1, ih + 1))
        roi[i] = (rng.integers(0, iw - w + 1), rng.integers(0, ih - h + 1), w, h)
        t, z = rng.uniform(-3.2, 3.2), rng.uniform(0.4, 1.3)
        affine[i] = (z * np.cos(t), z * np.sin(t), -z * np.sin(t), z * np.cos(t), rng.uniform(-9, 9), rng.uniform(-9, 9))
    for i in (0, n - 1):
        roi[i] = (0, 0, widths[i], heights[i])
    roi[n - 2] = (widths[n - 2] - 1, heights[n - 2] - 1, 1, 1)
    affine[0] = affine[n - 1] = (1, 0, 0, 1, 0, 0)          # every pixel, the last byte of the buffer among them
    affine[1] = (3.1, 0.4, -0.3, 2.9, 0.5, -0.5)            # rows wider than the usual LDS pitch
    affine[2] = (9.0, 4.0, -4.0, 9.0, 0.0, 0.0)             # boxes too large for LDS
    affine[3] = (1, 0, 0, 1, 5000, -5000)                   # nothing inside
    affine[4] = (np.nan, 0, 0, 1, 0, 0)
    return widths, heights, roi, affine


@pytest.mark.parametrize("layout,dtype", COMBOS)
@pytest.mark.parametrize("interp", [ops.LINEAR, ops.NEAREST])
@pytest.mark.parametrize("W,H", [(149, 90), (150, 90), (151, 90), (152, 90), (5, 7), (2, 2)])
@pytest.mark.parametrize("packed", [False, True])
def test_rows_at_every_phase(ctx, layout, dtype, interp, W, H, packed):
    import torch
    rng = np.random.default_rng(W * 100 + 10 * layout + dtype + (7 if packed else 0))
    n, OH, OW = 20, 75, 141
    img = rng.integers(0, 256, (n, H, W, 3), dtype=np.uint8)
    widths, heights, roi, affine = _batch(W, H, n, rng)
    if not packed:
        widths[:], heights[:] = W, H
    dw, dh = rng.integers(20, OW + 1, n).astype(np.uint32), rng.integers(10, OH + 1, n).astype(np.uint32)
    dw[5:14], dw[14], dw[0] = np.arange(1, 10), 35, OW
    wide = (W + 3) // 4 * 4
    ref_img = np.zeros((n, H, wide, 3), np.uint8)
    ref_img[:, :, :W] = img
    dd = ops.desc(n, OH, OW, layout, dtype)
    ref = ops.WarpAffine(ctx, ops.desc(n, H, wide, ops.NHWC, ops.UINT8), dd, interp)
    ref.update(roi, affine, dw, dh)
    assert ref.kernel_name == "rmx_warp_kernel(raw)", ref.plan
    want = ref.alloc_output(fill=5)
    ref.launch(torch.from_numpy(ref_img).cuda(), want)
    op = ops.WarpAffine(ctx, ops.desc(n, H, W, ops.NHWC, ops.UINT8), dd, interp)
    if packed:
        sizes = widths.astype(np.int64) * heights * 3
        offsets = (np.cumsum(sizes) - sizes).astype(np.uint64)
        src = torch.from_numpy(np.concatenate([img[i, :heights[i], :widths[i]].reshape(-1) for i in range(n)])).cuda()
        op.set_ragged_source(offsets, widths, heights, src.numel())
    else:
        src = torch.from_numpy(img).cuda()
    op.update(roi, affine, dw, dh)
    assert op.kernel_name == ("rmx_warp_kernel" if packed or W % 4 else "rmx_warp_kernel(raw)"), op.plan
    got = op.alloc_output(fill=5)
    op.launch(src, got)
    ctx.sync()
    got, want = got.cpu().numpy(), want.cpu().numpy()
    assert np.array_equal(got.view(np.uint8), want.view(np.uint8)), (op.plan, [i for i in range(n) if not np.array_equal(got[i], want[i], equal_nan=True)])
    if dtype == ops.UINT8:
        known = np.where(np.isnan(affine).any(1, keepdims=True), np.float32([1, 0, 0, 1, 5000, 5000]), affine)  # (the oracle takes numbers: no pixel inside)
        exp = orc.warp_affine(img, roi, np.stack([orc.affine_from_rocal(a) for a in known]), dw, dh, OH, OW, interp=interp)
        if layout == ops.NCHW:
            exp = exp.transpose(0, 3, 1, 2)
        keep = np.full_like(exp, 5)
        for i in range(n):
            x = (i, slice(None), slice(0, dh[i]), slice(0, dw[i])) if layout == ops.NCHW else (i, slice(0, dh[i]), slice(0, dw[i]))
            keep[x] = exp[x]
        assert np.array_equal(got, keep), (op.plan, [i for i in range(n) if not np.array_equal(got[i], keep[i])])
