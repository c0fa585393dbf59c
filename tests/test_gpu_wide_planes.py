"""Bilinear and nearest resizes to fp32 planes at the widths where a row is one tile or several (whole rows of up to 512 pixels where
their window fits LDS, 256 and less where it does not), mirrored, odd widths among them, bit for bit against the oracle."""
import numpy as np
import pytest

from oracle import orc
from rocal_amd import ops, workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("interp", [ops.LINEAR, ops.NEAREST])
@pytest.mark.parametrize("OW", [256, 257, 263, 299, 384, 511, 512, 513, 520])
@pytest.mark.parametrize("W", [640, 639])
def test_rows_of_one_tile_and_of_several(ctx, interp, OW, W):
    import torch
    rng = np.random.default_rng(OW + W)
    n, H, OH = 5, 60, 21
    img = rng.integers(0, 256, (n, H, W, 3), dtype=np.uint8)
    roi = np.array([[0, 0, W, H], [7, 3, 200, 50], [W - 101, 0, 101, 60], [1, 1, 333, 22], [5, 50, 634, 9]], np.uint32)
    dw, dh = np.array([OW, OW, OW - 1, OW // 2, OW], np.uint32), np.array([21, 5, 21, 20, 3], np.uint32)
    mirror = rng.integers(0, 2, n).astype(np.uint32)
    scale, bias = orc.cmn_scale_bias(wl.MEAN, wl.STD, n)
    exp = orc.resize(img, roi, dw, dh, OH, OW, interp=interp, mirror=mirror, scale=scale, bias=bias, layout=ops.NCHW, dtype=ops.FP32)
    op = ops.Resize(ctx, ops.desc(n, H, W, ops.NHWC, ops.UINT8), ops.desc(n, OH, OW, ops.NCHW, ops.FP32), interp)
    op.update_cmn(roi, dw, dh, scale, bias, mirror)
    out = op.alloc_output(fill=5)
    op.launch(torch.from_numpy(img).cuda(), out)
    ctx.sync()
    got = out.cpu().numpy()
    keep = np.full_like(exp, 5)
    for i in range(n):
        keep[i, :, :dh[i], :dw[i]] = exp[i, :, :dh[i], :dw[i]]
    assert np.array_equal(got.view(np.uint32), keep.view(np.uint32)), (op.plan, [i for i in range(n) if not np.array_equal(got[i], keep[i])])
