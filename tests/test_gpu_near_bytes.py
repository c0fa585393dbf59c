"""Nearest-pixel resizes of bytes to interleaved bytes, whose pixels are moved and not converted, against the oracle: rows of 1 to 17 pixels
and around tiles, mirrored and not, source rows at every phase, crops behind the resize."""
import numpy as np
import pytest

from oracle import orc
from rocal_amd import ops, workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W", [40, 41, 42, 43])
@pytest.mark.parametrize("widths", [(1, 2, 3, 7, 8, 9), (15, 16, 17, 24, 31, 33), (127, 128, 129, 256, 257, 263), (300, 511, 512, 513, 520, 64)])
def test_rows_of_every_width_mirrored_and_not(ctx, W, widths):
    import torch
    rng = np.random.default_rng(W + widths[0])
    n, H, OH, OW = 6, 21, 30, max(widths)
    img = rng.integers(0, 256, (n, H, W, 3), dtype=np.uint8)
    roi = np.array([[i % 3, i % 2, W - 3 - i, H - 2 - i] for i in range(n)], np.uint32)
    dw, dh = np.array(widths, np.uint32), np.array([30, 9, 1, 13, 30, 21], np.uint32)
    op = ops.Resize(ctx, ops.desc(n, H, W, ops.NHWC, ops.UINT8), ops.desc(n, OH, OW, ops.NHWC, ops.UINT8), ops.NEAREST)
    src = torch.from_numpy(img).cuda()
    for mirror in (np.zeros(n, np.uint32), np.ones(n, np.uint32), (np.arange(n) % 2).astype(np.uint32)):
        op.update(roi, dw, dh, mirror)
        out = op.alloc_output(fill=5)
        op.launch(src, out)
        ctx.sync()
        exp = orc.resize(img, roi, dw, dh, OH, OW, interp=orc.NEAREST, mirror=mirror, layout=ops.NHWC, dtype=ops.UINT8)
        want = np.full_like(exp, 5)
        for i in range(n):
            want[i, :dh[i], :dw[i]] = exp[i, :dh[i], :dw[i]]
        got = out.cpu().numpy()
        assert np.array_equal(got, want), "%d values differ (%s)" % (int((got != want).sum()), op.plan)
