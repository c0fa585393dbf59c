"""Normalize with the sample's own moments at the sizes where the moments pass can go wrong, bit for bit against the oracle: fewer
rows than workgroups per sample, rows of 1 to 9 pixels and of more groups than a workgroup has threads, windows on the last byte of
the buffer, a packed source, sums beyond 32 bits in one workgroup, and only the mean or only the deviation computed."""
import numpy as np
import pytest

from oracle import orc
from rocal_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w", [(1, 1), (3, 7), (5, 8), (9, 9), (8, 4200), (17, 63), (1100, 512)])
@pytest.mark.parametrize("mask", [3, 7])
@pytest.mark.parametrize("given", ["none", "mean", "stddev"])
def test_moments(ctx, h, w, mask, given):
    import torch
    rng = np.random.default_rng(h * 10000 + w + mask)
    n = 2
    img = rng.integers(0, 256, (n, h, w, 3), dtype=np.uint8)
    img[0] |= 0xc0  # (large sums)
    roi = np.array([[0, 0, w, h], [w // 3, h // 3, w - w // 3, h - h // 3]], np.uint32)
    kw = {"none": {}, "mean": dict(mean=[100.0, 90.0, 80.0]), "stddev": dict(stddev=[50.0, 60.0, 70.0])}[given]
    exp = orc.normalize(img, roi, axis_mask=mask, scale=1.5, shift=0.25, layout=ops.NCHW, dtype=ops.FP32, **kw)
    op = ops.Normalize(ctx, ops.desc(n, h, w, ops.NHWC, ops.UINT8), ops.desc(n, h, w, ops.NCHW, ops.FP32))
    packed = torch.from_numpy(np.concatenate([[0], img.reshape(-1)]).astype(np.uint8)).cuda()
    for ragged in (False, True):  # (ragged: image bases at odd addresses)
        if ragged:
            op.set_ragged_source(1 + np.arange(n, dtype=np.uint64) * h * w * 3, np.full(n, w), np.full(n, h), packed.numel())
        op.update(roi, axis_mask=mask, scale=1.5, shift=0.25, **kw)
        out = op.alloc_output()
        op.launch(packed if ragged else torch.from_numpy(img).cuda(), out)
        ctx.sync()
        got = out.cpu().numpy()
        for i in range(n):
            x = (slice(None), slice(0, roi[i, 3]), slice(0, roi[i, 2]))
            assert np.array_equal(got[i][x].view(np.uint32), exp[i][x].view(np.uint32)), (i, ragged)


@pytest.mark.parametrize("n,h,w,shares", [
    (1, 1, 8, "1x64"), (3, 32, 64, "1x64"), (1, 257, 8, "1x128"), (2, 2048, 7, "1x512"), (1, 2049, 8, "2x512"),  # wavefronts of 256 groups
    (1, 3, 32800, "8x512"), (1, 1030, 1024, "64x512"), (9, 1030, 1024, "32x512"), (65, 150, 1000, "8x512"), (200, 32, 32, "1x64")])
def test_moment_shares(ctx, n, h, w, shares):
    """Shares of a sample's moments: as many workgroups and wavefronts as its groups of 8 pixels keep busy, more of them in small
    batches; also more shares than rows."""
    import torch
    rng = np.random.default_rng(h + w)
    img = rng.integers(0, 256, (n, h, w, 3), dtype=np.uint8)
    img[0] |= 0xc0  # (large sums)
    roi = np.tile(np.array([0, 0, w, h], np.uint32), (n, 1))
    op = ops.Normalize(ctx, ops.desc(n, h, w, ops.NHWC, ops.UINT8), ops.desc(n, h, w, ops.NHWC, ops.FP16))
    op.update(roi, axis_mask=3, scale=1.5, shift=0.25)
    assert op.plan.endswith("moments=" + shares), op.plan
    out = op.alloc_output()
    op.launch(torch.from_numpy(img).cuda(), out)
    ctx.sync()
    exp = orc.normalize(img, roi, axis_mask=3, scale=1.5, shift=0.25, layout=ops.NHWC, dtype=ops.FP16)
    assert np.array_equal(out.cpu().numpy().view(np.uint16), exp.view(np.uint16))
