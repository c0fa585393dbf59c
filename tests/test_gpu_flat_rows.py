"""Whole frames walked as rows of 512 pixels at the frame sizes where that can go wrong, bit for bit against the oracle: one short
row, a last row of 1 to 8 pixels (which takes 8 of the row before), one exact row, frames of odd byte counts, destinations off
16-byte alignment; the bytes around the destination must stay as they were."""
import numpy as np
import pytest

from oracle import orc
from rocal_amd import ops

pytestmark = pytest.mark.gpu
COMBOS = [(ops.NCHW, ops.FP16), (ops.NCHW, ops.FP32), (ops.NCHW, ops.UINT8), (ops.NHWC, ops.FP16), (ops.NHWC, ops.FP32), (ops.NHWC, ops.UINT8)]
SIZES = [(1, 8), (1, 11), (7, 73), (2, 256), (3, 171), (5, 103), (8, 65), (24, 64), (31, 33), (1, 1537), (40, 52)]


@pytest.mark.parametrize("layout,dtype", COMBOS)
@pytest.mark.parametrize("h,w", SIZES)
def test_frames_of_any_size(ctx, h, w, layout, dtype):
    import torch
    n = 3
    rng = np.random.default_rng(h * 4000 + w + 10 * layout + dtype)
    img, img2 = (rng.integers(0, 256, (n, h, w, 3), dtype=np.uint8) for _ in range(2))
    roi = np.tile(np.array([0, 0, w, h], np.uint32), (n, 1))
    f = lambda lo, hi: rng.uniform(lo, hi, n).astype(np.float32)  # noqa: E731
    alpha, beta, hue, sat, gamma, ratio = f(0.6, 1.4), f(-20, 20), f(-180, 180), f(0.2, 1.8), f(0.3, 3.0), f(0.0, 1.0)
    scale, bias = rng.uniform(0.5, 1.5, (n, 3)).astype(np.float32), rng.integers(-20, 20, (n, 3)).astype(np.float32)
    kw = dict(layout=layout, dtype=dtype)
    no_mirror = np.zeros(n, np.uint32)
    cases = [
        (ops.ColorTwist, lambda op: op.update(roi, alpha, beta, hue, sat), (img,), orc.color_twist(img, roi, alpha, beta, hue, sat, **kw)),
        (ops.Brightness, lambda op: op.update(roi, alpha, beta), (img,), orc.brightness(img, roi, alpha, beta, **kw)),
        (ops.Gamma, lambda op: op.update(roi, gamma), (img,), orc.gamma(img, roi, gamma, **kw)),
        (ops.Blend, lambda op: op.update(roi, ratio), (img, img2), orc.blend(img, img2, roi, ratio, **kw)),
        (ops.CropMirrorNormalize, lambda op: op.update(roi, scale, bias, no_mirror), (img,),
         orc.crop_mirror_normalize(img, roi, scale, bias, no_mirror, h, w, layout, dtype)),
    ]
    for cls, update, srcs, exp in cases:
        op = cls(ctx, ops.desc(n, h, w, ops.NHWC, ops.UINT8), ops.desc(n, h, w, layout, dtype))
        update(op)
        assert "flat_rows=%d" % (-(-h * w // 512)) in op.plan, op.plan
        esz = exp.dtype.itemsize
        for shift in (0, 1):
            raw = torch.full((exp.size * esz + 64,), 0x5A, dtype=torch.uint8, device="cuda")
            out = raw[shift * esz: shift * esz + exp.size * esz].view(ops.torch_dtype(dtype)).view(exp.shape)
            op.launch(*[torch.from_numpy(s).cuda() for s in srcs], out)
            ctx.sync()
            assert np.array_equal(out.cpu().numpy().view(np.uint8), exp.view(np.uint8)), (cls.__name__, shift, op.plan)
            r = raw.cpu().numpy()
            assert (r[:shift * esz] == 0x5A).all() and (r[shift * esz + exp.size * esz:] == 0x5A).all(), (cls.__name__, shift)
