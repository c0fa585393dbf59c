"""Windows that read the first and the last bytes of the batch buffer, at every length that a row can have past whole 16-byte pieces:
resizes (linear, nearest, triangular) and warps of one and two whole images, a few rows high and more, padded (row strides of
every remainder mod 4) and packed into a buffer that ends with the last image's last byte. Bytes against the oracle."""
import numpy as np
import pytest

from oracle import orc
from rocal_amd import ops

pytestmark = pytest.mark.gpu


def _source(op, img, packed):
    import torch
    n, h, w = img.shape[:3]
    if not packed:
        return torch.from_numpy(img).cuda()
    op.set_ragged_source(np.arange(n, dtype=np.uint64) * (h * w * 3), np.full(n, w, np.uint32), np.full(n, h, np.uint32), img.size)
    return torch.from_numpy(img.reshape(-1)).cuda()


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("n,h", [(1, 1), (1, 3), (2, 17), (1, 50)])
@pytest.mark.parametrize("width", list(range(37, 54)) + [5, 1])
def test_last_bytes(ctx, width, n, h, packed):
    rng = np.random.default_rng(width * 100 + h)
    img = rng.integers(0, 256, (n, h, width, 3), dtype=np.uint8)
    roi = np.tile(np.array([0, 0, width, h], np.uint32), (n, 1))
    sd = ops.desc(n, h, width, ops.NHWC, ops.UINT8)
    got, want = {}, {}
    for name, interp, (oh, ow) in (("linear", ops.LINEAR, (23, 40)), ("linear, odd", ops.LINEAR, (9, 77)), ("nearest", ops.NEAREST, (23, 40)),
                                   ("triangular", ops.TRIANGULAR, (max(1, h // 2), max(1, width // 2))), ("triangular, larger", ops.TRIANGULAR, (h + h // 2, width + 9))):
        op = ops.Resize(ctx, sd, ops.desc(n, oh, ow, ops.NHWC, ops.UINT8), interp)
        src = _source(op, img, packed)
        dw, dh = np.full(n, ow, np.uint32), np.full(n, oh, np.uint32)
        op.update(roi, dw, dh)
        got[name] = op.alloc_output(fill=3)
        op.launch(src, got[name])
        want[name] = orc.resize(img, roi, dw, dh, oh, ow, interp=interp, layout=ops.NHWC, dtype=ops.UINT8)
    dw, dh = np.full(n, width, np.uint32), np.full(n, h, np.uint32)
    for interp in (ops.LINEAR, ops.NEAREST):
        for what, a in (("same", (1, 0, 0, 1, 0, 0)), ("turned", (0.8, 0.6, -0.6, 0.8, 1.5, -2.0)), ("upside down", (-1, 0, 0, -1, 0, 0))):
            name = "warp %d %s" % (interp, what)
            affine = np.tile(np.array(a, np.float32), (n, 1))
            op = ops.WarpAffine(ctx, sd, sd, interp)
            src = _source(op, img, packed)
            op.update(roi, affine, dw, dh)
            got[name] = op.alloc_output(fill=3)
            op.launch(src, got[name])
            want[name] = orc.warp_affine(img, roi, np.stack([orc.affine_from_rocal(v) for v in affine]), dw, dh, h, width, interp=interp)
    ctx.sync()
    for name in got:
        g = got[name].cpu().numpy()
        assert np.array_equal(g, want[name]), "%s: %d values differ" % (name, int((g != want[name]).sum()))
