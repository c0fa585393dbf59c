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
