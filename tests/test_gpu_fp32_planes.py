"""fp32 planes of the streaming resize kernels, whose rows' lanes exchange their runs through LDS: whole groups of 8, and behind a colour
twist every width that is a multiple of 4 (a last run that overlaps its neighbour, rows of one and two pieces per lane, x-tiles),
samples narrower than the destination, mirrored and not, destinations at a 16-byte piece and at single elements. Every value
against the oracle, and the destination outside the written windows against what it held."""
import numpy as np
import pytest

from oracle import orc
from rocal_amd import ops, workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("twist", [False, True])
@pytest.mark.parametrize("width", [4, 8, 12, 20, 36, 64, 100, 128, 132, 252, 260, 300, 384, 516, 1028, 301])
@pytest.mark.parametrize("source_width", [96, 97])
def test_planes_of_every_kind(ctx, width, source_width, twist):
    import torch
    rng = np.random.default_rng(width * 10 + twist)
    n, H, oh = 4, 40, 13
    img = wl.smooth_noise(rng, n, H, source_width, sigma=1.0)
    roi = np.array([[0, 0, source_width, H], [1, 2, 70, 30], [source_width - 41, H - 9, 41, 9], [3, 0, 90, H]], np.uint32)
    rw = np.array([width, width, max(4, width - 4), max(4, width // 2 // 4 * 4)], np.uint32)
    rh = np.array([oh, oh - 1, oh, 5], np.uint32)
    mirror = np.array([0, 1, 1, 0], np.uint32)
    scale, bias = orc.cmn_scale_bias(wl.MEAN, wl.STD, n)
    colour = [rng.uniform(*r, n).astype(np.float32) for r in ((0.6, 1.4), (-20, 20), (-90, 90), (0.5, 1.5))]
    mid = orc.resize(img, roi, rw, rh, oh, width, interp=orc.LINEAR)
    whole = np.stack([np.zeros(n), np.zeros(n), rw, rh], -1).astype(np.uint32)
    exp = orc.crop_mirror_normalize(orc.color_twist(mid, whole, *colour) if twist else mid, whole, scale, bias, mirror, oh, width, orc.NCHW, orc.FP32)
    op = ops.Resize(ctx, ops.desc(n, H, source_width, ops.NHWC, ops.UINT8), ops.desc(n, oh, width, ops.NCHW, ops.FP32), ops.LINEAR,
                    flags=ops.F_QUANTIZE_U8 | (ops.F_COLOR_TWIST if twist else 0))
    if twist:
        op.update_color_cmn(roi, rw, rh, scale, bias, colour, mirror)
    else:
        op.update_cmn(roi, rw, rh, scale, bias, mirror)
    src = torch.from_numpy(img).cuda()
    size = n * 3 * oh * width
    for shift in (0, 4, 1):  # elements behind an aligned address
        buf = torch.full((size + 8,), 7.0, dtype=torch.float32, device="cuda")
        op.launch(src, buf[shift:shift + size])
        ctx.sync()
        got = buf.cpu().numpy()
        want = np.full(size + 8, 7.0, np.float32)
        view = want[shift:shift + size].reshape(n, 3, oh, width)
        for i in range(n):
            view[i, :, :rh[i], :rw[i]] = exp[i, :, :rh[i], :rw[i]]
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), "shift %d (%s): %d values differ" % (shift, op.plan, int((got != want).sum()))


@pytest.mark.parametrize("twist", [False, True])
@pytest.mark.parametrize("layout", [ops.NCHW, ops.NHWC])
@pytest.mark.parametrize("source_width", [96, 97])
@pytest.mark.parametrize("width", [64, 72, 100, 101])
def test_room_for_the_exchange_where_there_is_one(ctx, width, source_width, layout, twist):
    """The LDS slice of an fp32 plan against the half-precision one's: as large but for the slab of kernels that exchange their runs."""
    n, H, oh = 3, 40, 20
    roi = np.tile(np.array([0, 0, source_width, H], np.uint32), (n, 1))
    rw, rh = np.full(n, width, np.uint32), np.full(n, oh, np.uint32)
    scale, bias = orc.cmn_scale_bias(wl.MEAN, wl.STD, n)
    lds = {}
    for dtype in (ops.FP32, ops.FP16):
        op = ops.Resize(ctx, ops.desc(n, H, source_width, ops.NHWC, ops.UINT8), ops.desc(n, oh, width, layout, dtype), ops.LINEAR,
                        flags=ops.F_QUANTIZE_U8 | (ops.F_COLOR_TWIST if twist else 0))
        if twist:
            op.update_color_cmn(roi, rw, rh, scale, bias, [np.full(n, v, np.float32) for v in (1.1, 2.0, 30.0, 0.9)], None)
        else:
            op.update_cmn(roi, rw, rh, scale, bias, None)
        lds[dtype] = int(dict(p.split("=") for p in op.plan.split())["lds_per_wave"])
    whole, one_phase = width % 8 == 0, source_width % 4 == 0
    exchange = layout == ops.NHWC or (whole and one_phase) or (twist and width % 4 == 0)
    assert lds[ops.FP32] - lds[ops.FP16] == (0 if not exchange else 2048 if layout == ops.NCHW else 6144), (lds, op.plan)
