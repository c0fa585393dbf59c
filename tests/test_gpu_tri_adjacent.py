"""The streaming triangular kernel whose lanes own neighbouring columns, bit for bit against the oracle, where it can go wrong: rows at every
byte phase (padded and packed images), windows that grow by any ratio and those that shrink in one batch, clamped taps at all four
edges, rows of two and three pixels, a last tile of one column, mirrors, crops behind the resize, strips of every length, and windows
whose rounding gives a source row to three output rows (the third starts its accumulators from it)."""
import numpy as np
import pytest

from oracle import orc
from rocal_amd import ops, workloads as wl

pytestmark = pytest.mark.gpu

FORMATS = [(ops.NCHW, ops.FP16), (ops.NCHW, ops.FP32), (ops.NCHW, ops.UINT8), (ops.NHWC, ops.FP16), (ops.NHWC, ops.FP32), (ops.NHWC, ops.UINT8)]


def _check(c, img, roi, dw, dh, OH, OW, layout, dtype, mirror, packed=None, quant=False, kernel="rmx_resize_tri_adj_kernel"):
    import torch
    n, H, W = img.shape[:3]
    norm = dtype != ops.UINT8
    s, b = orc.cmn_scale_bias(wl.MEAN, wl.STD, n)
    op = ops.Resize(c, ops.desc(n, H, W, ops.NHWC, ops.UINT8), ops.desc(n, OH, OW, layout, dtype), ops.TRIANGULAR, flags=ops.F_QUANTIZE_U8 if quant else 0)
    src = img
    if packed is not None:
        src, offsets, strides, widths, heights = packed
        op.set_ragged_source(offsets, widths, heights, src.size, row_strides=strides)
    if norm:
        op.update_cmn(roi, dw, dh, s, b, mirror)
    else:
        op.update(roi, dw, dh, mirror)
    assert op.kernel_name == kernel and ("adjacent=1" in op.plan) == (kernel == "rmx_resize_tri_adj_kernel"), (op.kernel_name, op.plan)
    out = op.alloc_output(fill=6)
    op.launch(torch.from_numpy(np.ascontiguousarray(src)).cuda(), out)
    c.sync()
    got = out.cpu().numpy()
    exp = orc.resize(img, roi, dw, dh, OH, OW, interp=orc.TRIANGULAR, mirror=mirror, scale=s if norm else None, bias=b if norm else None, layout=layout, dtype=dtype,
                     flags=orc.F_QUANTIZE_U8 if quant else 0)
    want = np.full_like(exp, 6)
    for i in range(n):
        if layout == ops.NCHW:
            want[i, :, :dh[i], :dw[i]] = exp[i, :, :dh[i], :dw[i]]
        else:
            want[i, :dh[i], :dw[i]] = exp[i, :dh[i], :dw[i]]
    for i in range(n):
        assert np.array_equal(np.ascontiguousarray(got[i]).view(np.uint8), np.ascontiguousarray(want[i]).view(np.uint8)), "sample %d: %d values differ (%s)" % (
            i, int((got[i] != want[i]).sum()), op.plan)


def _batch(seed, W):
    """Twelve windows of a W-pixel-wide source: growing by up to 16, shrinking by up to 4, both, at every edge; widths 2 to 130."""
    rng = np.random.default_rng(seed)
    H, OH, OW = 150, 96, 130
    dw = np.array([130, 129, 96, 2, 3, 64, 127, 128, 5, 130, 100, 31], np.uint32)
    dh = np.array([96, 90, 96, 96, 7, 96, 95, 96, 1, 96, 60, 96], np.uint32)
    sw = np.minimum(np.array([W, 40, 9, 2, 12, 100, 130, W, 3, 17, W, 31], np.uint32), W)
    sh = np.array([6, 30, 150, 1, 20, 95, 40, 144, 3, 24, 150, 2], np.uint32)
    x = np.array([0, W - sw[1], 3, W - sw[3], 1, 2, 0, 0, W - 3, 5, 0, W - sw[11]], np.uint32)
    x = np.minimum(x, W - sw)
    y = np.minimum(np.array([0, 120, 0, 149, 130, 55, 1, 3, 147, 0, 0, 148], np.uint32), H - sh)
    img = wl.smooth_noise(rng, len(dw), H, W, sigma=1.0)
    return img, np.stack([x, y, sw, sh], 1).astype(np.uint32), dw, dh, OH, OW, (np.arange(len(dw)) % 2).astype(np.uint32)


@pytest.mark.parametrize("layout,dtype", FORMATS)
@pytest.mark.parametrize("W", [132, 133, 134, 135])
def test_rows_at_every_phase_ratios_and_widths(ctx, layout, dtype, W):
    img, roi, dw, dh, OH, OW, mirror = _batch(W, W)
    _check(ctx, img, roi, dw, dh, OH, OW, layout, dtype, mirror)


@pytest.mark.parametrize("layout,dtype", [f for f in FORMATS if f[1] != ops.UINT8])
@pytest.mark.parametrize("W", [132, 133])
def test_quantised(ctx, layout, dtype, W):
    """As a resize node that has taken in the normalisation behind it asks for: rounded to bytes, then normalised."""
    img, roi, dw, dh, OH, OW, mirror = _batch(W + 7, W)
    _check(ctx, img, roi, dw, dh, OH, OW, layout, dtype, mirror, quant=True)


@pytest.mark.parametrize("W,grow,kernel", [(132, 90, "rmx_resize_tri_dma_kernel"), (133, 90, "rmx_resize_tri_kernel"), (132, 20, "rmx_resize_tri_kernel")])
def test_a_sample_of_one_pixel_rows_sends_its_batch_to_another_kernel(ctx, W, grow, kernel):
    """No lane has two columns there: eight accumulator sets where rows start at one phase and no window grows by more than they allow."""
    rng = np.random.default_rng(W + grow)
    n, H, OH, OW = 4, 150, 120, 64
    img = rng.integers(0, 256, (n, H, W, 3), dtype=np.uint8)
    roi = np.array([[0, 0, W, H], [5, 7, 60, grow], [9, 1, 4, 100], [0, 0, 3, H]], np.uint32)
    dw, dh = np.array([64, 33, 1, 1], np.uint32), np.array([120, 120, 90, 120], np.uint32)
    for layout, dtype in ((ops.NCHW, ops.FP16), (ops.NHWC, ops.FP32)):
        _check(ctx, img, roi, dw, dh, OH, OW, layout, dtype, np.array([0, 1, 1, 0], np.uint32), kernel=kernel)


@pytest.mark.parametrize("rows", [4, 5, 23, 64])
def test_strips_of_every_length(rows):
    from conftest import _ctx_with_env
    c = _ctx_with_env(RMX_TUNE_TRI_ROWS=rows)
    try:
        img, roi, dw, dh, OH, OW, mirror = _batch(rows, 133)
        _check(c, img, roi, dw, dh, OH, OW, ops.NCHW, ops.FP16, mirror)
        _check(c, img, roi, dw, dh, OH, OW, ops.NHWC, ops.FP32, 1 - mirror)
    finally:
        c.close()


@pytest.mark.parametrize("tight", [False, True])
def test_packed_images_of_odd_widths(ctx, tight):
    """Images one behind the other, rows of any number of bytes, the last window's rows on the buffer's last bytes; one of them so narrow that
    its rows' pieces reach over several rows."""
    rng = np.random.default_rng(5)
    widths, heights = np.array([77, 50, 5, 129, 3], np.uint32), np.array([60, 41, 30, 77, 9], np.uint32)
    strides = (widths * 3 + (0 if tight else 5)).astype(np.uint32)
    n, H, W = len(widths), int(heights.max()), int(widths.max())
    img = np.zeros((n, H, W, 3), np.uint8)
    buf, offsets = [np.zeros(3, np.uint8)], []
    for i in range(n):
        h, w = int(heights[i]), int(widths[i])
        img[i, :h, :w] = rng.integers(0, 256, (h, w, 3), dtype=np.uint8)
        rows = np.full((h, int(strides[i])), 0xEE, np.uint8)
        rows[:, :3 * w] = img[i, :h, :w].reshape(h, 3 * w)
        offsets.append(sum(len(b) for b in buf))
        buf.append(rows.reshape(-1)[:(h - 1) * int(strides[i]) + 3 * w] if i == n - 1 else rows.reshape(-1))
    src = np.concatenate(buf)
    roi = np.stack([np.zeros(n), np.zeros(n), widths, heights], 1).astype(np.uint32)
    dw, dh = np.array([40, 70, 20, 64, 6], np.uint32), np.array([33, 70, 50, 40, 70], np.uint32)
    _check(ctx, img, roi, dw, dh, 70, 70, ops.NCHW, ops.FP16, np.array([0, 1, 0, 1, 1], np.uint32), (src, np.array(offsets, np.uint64), strides, widths, heights))


# source rows, output rows, first source row: rounding makes a coefficient of a third output row a little more than 0
TWICE = [(430, 290, 135), (390, 330, 134), (212, 116, 14), (205, 145, 72)]


def _third_rows(sh, dh, y0):
    """How many source rows have a coefficient other than 0 in three output rows, by the fp32 law."""
    f = np.float32
    ry = f(f(sh) / f(dh))
    raw = (np.arange(dh).astype(f) * ry + f(f(f(ry - f(1)) * f(0.5)) - ry)).astype(f) + f(y0)
    loc = np.ceil(raw)
    k = np.arange(int(np.ceil(2 * ry))).astype(f)
    c = f(1) - np.abs((((loc - raw).astype(f) - ry)[:, None] + k) * f(f(1) / ry))
    rows = np.clip(loc[:, None] + k, y0, y0 + sh - 1)
    first, last = np.where(c > 0, rows, np.inf).min(1), np.where(c > 0, rows, -np.inf).max(1)
    return int((first[2:] <= last[:-2]).sum())


@pytest.mark.parametrize("rows", [0, 64])
def test_source_rows_of_three_output_rows(rows):
    assert all(_third_rows(*t) for t in TWICE)
    from conftest import _ctx_with_env
    c = _ctx_with_env(RMX_TUNE_TRI_ROWS=rows)
    rng = np.random.default_rng(11)
    n, H, W = len(TWICE) + 1, 570, 61
    img = rng.integers(0, 256, (n, H, W, 3), dtype=np.uint8)
    roi = np.array([[2, y0, 55, sh] for sh, _, y0 in TWICE] + [[0, 0, 40, 20]], np.uint32)
    dh = np.array([d for _, d, _ in TWICE] + [90], np.uint32)
    dw = np.array([40, 55, 31, 20, 50], np.uint32)
    try:
        _check(c, img, roi, dw, dh, int(dh.max()), 55, ops.NCHW, ops.FP32, np.array([0, 1, 0, 1, 0], np.uint32))
        _check(c, img, roi, dw, dh, int(dh.max()), 55, ops.NHWC, ops.UINT8, np.array([1, 0, 0, 1, 0], np.uint32))
    finally:
        c.close()


# ratios at which that happens every few rows: 11/7, 3.4
OFTEN = [(550, 350, 0), (476, 140, 7), (352, 224, 200), (330, 210, 61), (352, 224, 0)]


@pytest.mark.parametrize("rows", [0, 7, 64])
@pytest.mark.parametrize("W,layout,dtype", [(140, ops.NCHW, ops.FP16), (141, ops.NCHW, ops.FP16), (141, ops.NHWC, ops.FP32), (140, ops.NHWC, ops.UINT8)])
def test_ratios_whose_rows_meet_again_and_again(rows, W, layout, dtype):
    """Strips in which many output rows start their accumulators from a source row that they share: 12 to 64 output rows of 2 to 4 source
    rows each (the table of coefficients is made again on the way, also right at such rows), horizontal taps of every number."""
    assert all(_third_rows(*t) > 2 for t in OFTEN)
    from conftest import _ctx_with_env
    c = _ctx_with_env(RMX_TUNE_TRI_ROWS=rows)
    rng = np.random.default_rng(W + rows)
    n, H = len(OFTEN), 560
    img = rng.integers(0, 256, (n, H, W, 3), dtype=np.uint8)
    roi = np.array([[i, y0, W - 3 - i, sh] for i, (sh, _, y0) in enumerate(OFTEN)], np.uint32)
    dh = np.array([d for _, d, _ in OFTEN], np.uint32)
    dw = np.array([130, 100, 70, 46, 36], np.uint32)
    try:
        _check(c, img, roi, dw, dh, int(dh.max()), 130, layout, dtype, np.array([0, 1, 0, 1, 0], np.uint32))
    finally:
        c.close()
