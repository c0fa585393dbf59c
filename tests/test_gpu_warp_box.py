"""Boxes of a warp's tiles about the pitches that its LDS rows have (10 and 11 pieces of 16 bytes, more), without a spare row or column:
maps that keep, shrink by a little and shrink by more, at angles about the axes and between them, windows inside an image and on its
edges, shifts that push tiles across every side of the window and just outside it. Bytes against the oracle."""
import numpy as np
import pytest

from oracle import orc
from rocal_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [200, 201])  # rows at one byte phase, at every phase
@pytest.mark.parametrize("interp", [ops.LINEAR, ops.NEAREST])
@pytest.mark.parametrize("shrink", [1.0, 1.03, 1.06, 1.1, 1.111, 1.16, 1.25, 1.45, 1.6])
def test_boxes(ctx, shrink, interp, width):
    import torch
    H, n = 180, 24
    rng = np.random.default_rng(int(shrink * 1000) + width)
    img = rng.integers(0, 256, (n, H, width, 3), dtype=np.uint8)
    roi, affine = np.empty((n, 4), np.uint32), np.empty((n, 6), np.float32)
    for i in range(n):
        w, h = (width, H) if i % 3 == 0 else (int(rng.integers(1, width + 1)), int(rng.integers(1, H + 1)))
        roi[i] = (rng.integers(0, width - w + 1), rng.integers(0, H - h + 1), w, h)
        angle = (0.0, np.pi / 2, np.pi / 4, np.pi / 6, -np.pi / 6, np.pi, rng.uniform(-3, 3), rng.uniform(-0.1, 0.1))[i % 8]
        c, s = shrink * np.cos(angle), shrink * np.sin(angle)
        far = rng.choice([0.0, 0.25, 16.0, w / 2 + 1, -w / 2 - 1, h / 2 + 0.5, -h / 2 - 33], 2) if i else (0.0, 0.0)
        affine[i] = (c, s, -s, c, far[0], far[1])
    roi[n - 1] = (0, 0, width, H)  # (with the buffer's last byte)
    dw, dh = np.full(n, width, np.uint32), np.full(n, H, np.uint32)
    sd = ops.desc(n, H, width, ops.NHWC, ops.UINT8)
    op = ops.WarpAffine(ctx, sd, sd, interp)
    op.update(roi, affine, dw, dh)
    assert op.kernel_name == ("rmx_warp_kernel" if width % 4 else "rmx_warp_kernel(raw)")
    got = op.alloc_output(fill=3)
    op.launch(torch.from_numpy(img).cuda(), got)
    ctx.sync()
    want = orc.warp_affine(img, roi, np.stack([orc.affine_from_rocal(a) for a in affine]), dw, dh, H, width, interp=interp)
    got = got.cpu().numpy()
    assert np.array_equal(got, want), [(i, int((got[i] != want[i]).sum())) for i in range(n) if not np.array_equal(got[i], want[i])]


@pytest.mark.parametrize("width", [200, 201])
@pytest.mark.parametrize("interp", [ops.LINEAR, ops.NEAREST])
@pytest.mark.parametrize("rows", [1, 2, 3])
def test_windows_of_few_rows_at_the_buffers_end(ctx, rows, interp, width):
    """Maps that leave tiles less than a row above such a window, beside it and below it."""
    import torch
    H, dh = 60, 64
    rng = np.random.default_rng(width + rows)
    affine = np.array([(1, 0, 0, 1, 0, s) for s in (0, -0.5, 0.25, 1, -1, 25, -25.5, 31.5, -31.75)] +
                      [(0.98, 0.2, -0.2, 0.98, x, s) for x, s in ((0, 0.5), (60, 9), (-60, -9.5))], np.float32)
    n = len(affine)
    for height in (H, rows):  # the last rows of images, images of these rows
        img = rng.integers(0, 256, (n, height, width, 3), dtype=np.uint8)
        roi = np.tile(np.array([0, height - rows, width, rows], np.uint32), (n, 1))
        dw, dhs = np.full(n, width, np.uint32), np.full(n, dh, np.uint32)
        op = ops.WarpAffine(ctx, ops.desc(n, height, width, ops.NHWC, ops.UINT8), ops.desc(n, dh, width, ops.NHWC, ops.UINT8), interp)
        for first in range(n):  # (every map at the end of the buffer once)
            a = np.roll(affine, first, axis=0)
            op.update(roi, a, dw, dhs)
            got = op.alloc_output(fill=3)
            op.launch(torch.from_numpy(img).cuda(), got)
            ctx.sync()
            want = orc.warp_affine(img, roi, np.stack([orc.affine_from_rocal(v) for v in a]), dw, dhs, dh, width, interp=interp)
            got = got.cpu().numpy()
            assert np.array_equal(got, want), [(i, int((got[i] != want[i]).sum())) for i in range(n) if not np.array_equal(got[i], want[i])]
