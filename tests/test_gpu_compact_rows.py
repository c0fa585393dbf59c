"""Parameter rows that travel in the kernel's arguments against the same rows in a device table, bit for bit: every kind of record
(windows with mirrors and x-tiles, colour factors, matrices, the order of a sorted batch, a packed source's layout), batch sizes at
which the records just fit and just do not, and coordinates beyond what a record can hold."""
import numpy as np
import pytest

from oracle import orc
from rocal_amd import ops, workloads as wl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx_table():
    from conftest import _ctx_with_env
    c = _ctx_with_env(RMX_TUNE_COMPACT=0)
    yield c
    c.sync()


def _windows(rng, n, h, w, lo):
    ww, hh = rng.integers(lo, w + 1, n), rng.integers(lo, h + 1, n)
    return np.stack([rng.integers(0, w - ww + 1), rng.integers(0, h - hh + 1), ww, hh], axis=1).astype(np.uint32)


def _resize(c, rng_seed, n, interp, packed=False, chain=False):
    rng = np.random.default_rng(rng_seed)
    h, w, o = 40, 56, 24
    flags = (ops.F_QUANTIZE_U8 | (ops.F_COLOR_TWIST if chain else 0)) if interp == ops.LINEAR else 0
    op = ops.Resize(c, ops.desc(n, h, w, ops.NHWC, ops.UINT8), ops.desc(n, o, o, ops.NCHW, ops.FP16), interp, flags=flags)
    img = rng.integers(0, 256, (n, h, w, 3), dtype=np.uint8)
    roi, d = _windows(rng, n, h, w, 9), np.full(n, o, np.uint32)
    scale, bias = orc.cmn_scale_bias(wl.MEAN, wl.STD, n)
    mirror = rng.integers(0, 2, n).astype(np.uint32)
    if packed:
        W, H = np.full(n, w, np.uint32), np.full(n, h, np.uint32)
        op.set_ragged_source(np.arange(n, dtype=np.uint64) * h * w * 3, W, H, n * h * w * 3)
    if chain:
        f = lambda lo, hi: rng.uniform(lo, hi, n).astype(np.float32)  # noqa: E731
        op.update_color_cmn(roi, d, d, scale, bias, (f(0.7, 1.3), f(-9, 9), f(-30, 30), f(0.5, 1.5)), mirror)
    else:
        op.update_cmn(roi, d, d, scale, bias, mirror)
    return op, img


def _resize_crops(c, seed, n, interp, packed=False, chain=False, o=37):
    """Resized images of one size of which every sample writes a window of its own size, odd ones and one-pixel ones among them."""
    rng = np.random.default_rng(seed)
    h, w = 40, 56
    flags = (ops.F_QUANTIZE_U8 | (ops.F_COLOR_TWIST if chain else 0)) if interp == ops.LINEAR else 0
    op = ops.Resize(c, ops.desc(n, h, w, ops.NHWC, ops.UINT8), ops.desc(n, o, o, ops.NCHW, ops.FP32), interp, flags=flags)
    roi, d = _windows(rng, n, h, w, 9), np.full(n, o, np.uint32)
    scale, bias = orc.cmn_scale_bias(wl.MEAN, wl.STD, n)
    crop, mirror = _windows(rng, n, o, o, 1), rng.integers(0, 2, n).astype(np.uint32)
    if packed:
        W, H = np.full(n, w, np.uint32), np.full(n, h, np.uint32)
        op.set_ragged_source(np.arange(n, dtype=np.uint64) * h * w * 3, W, H, n * h * w * 3)
    if chain:
        f = lambda lo, hi: rng.uniform(lo, hi, n).astype(np.float32)  # noqa: E731
        op.update_color_cmn(roi, d, d, scale, bias, (f(0.7, 1.3), f(-9, 9), f(-30, 30), f(0.5, 1.5)), mirror, crop_roi=crop)
    else:
        op.update_cmn(roi, d, d, scale, bias, mirror, crop_roi=crop)
    return op, rng.integers(0, 256, (n, h, w, 3), dtype=np.uint8)


def _crop(c, seed, n):
    rng = np.random.default_rng(seed)
    op = ops.CropMirrorNormalize(c, ops.desc(n, 30, 40, ops.NHWC, ops.UINT8), ops.desc(n, 24, 33, ops.NCHW, ops.FP32))
    scale, bias = orc.cmn_scale_bias(wl.MEAN, wl.STD, n)
    op.update(_windows(rng, n, 24, 33, 8), scale, bias, rng.integers(0, 2, n).astype(np.uint32))
    return op, rng.integers(0, 256, (n, 30, 40, 3), dtype=np.uint8)


def _flip(c, seed, n):
    rng = np.random.default_rng(seed)
    sd = ops.desc(n, 21, 35, ops.NHWC, ops.UINT8)
    op = ops.Flip(c, sd, sd)
    op.update(_windows(rng, n, 21, 35, 8), rng.integers(0, 2, n), rng.integers(0, 2, n))
    return op, rng.integers(0, 256, (n, 21, 35, 3), dtype=np.uint8)


def _twist(c, seed, n, roi=False):
    rng = np.random.default_rng(seed)
    sd = ops.desc(n, 18, 26, ops.NHWC, ops.UINT8)
    op = ops.ColorTwist(c, sd, sd)
    f = lambda lo, hi: rng.uniform(lo, hi, n).astype(np.float32)  # noqa: E731
    win = _windows(rng, n, 18, 26, 8) if roi else np.tile(np.array([0, 0, 26, 18], np.uint32), (n, 1))
    op.update(win, f(0.5, 1.5), f(-9, 9), f(-30, 30), f(0.5, 1.5))
    return op, rng.integers(0, 256, (n, 18, 26, 3), dtype=np.uint8)


def _brightness(c, seed, n):
    rng = np.random.default_rng(seed)
    sd = ops.desc(n, 18, 26, ops.NHWC, ops.UINT8)
    op = ops.Brightness(c, sd, sd)
    op.update(np.tile(np.array([0, 0, 26, 18], np.uint32), (n, 1)), rng.uniform(0.5, 1.5, n), np.full(n, 3.0))
    return op, rng.integers(0, 256, (n, 18, 26, 3), dtype=np.uint8)


def _rotate(c, seed, n, roi=False):
    rng = np.random.default_rng(seed)
    sd = ops.desc(n, 36, 44, ops.NHWC, ops.UINT8)
    op = ops.Rotate(c, sd, sd)
    win = _windows(rng, n, 36, 44, 8) if roi else np.tile(np.array([0, 0, 44, 36], np.uint32), (n, 1))
    op.update(win, rng.uniform(-90, 90, n), np.full(n, 44), np.full(n, 36))
    return op, rng.integers(0, 256, (n, 36, 44, 3), dtype=np.uint8)


# (maker, dwords of a record): 768 dwords of records fit
MAKERS = {
    "resize": (lambda c, s, n: _resize(c, s, n, ops.LINEAR), 2),
    "resize packed": (lambda c, s, n: _resize(c, s, n, ops.LINEAR, packed=True), 4),
    "chain": (lambda c, s, n: _resize(c, s, n, ops.LINEAR, chain=True), 6),
    "nearest": (lambda c, s, n: _resize(c, s, n, ops.NEAREST), 2),
    "triangular": (lambda c, s, n: _resize(c, s, n, ops.TRIANGULAR), 3),
    "triangular packed": (lambda c, s, n: _resize(c, s, n, ops.TRIANGULAR, packed=True), 5),
    "resize crops": (lambda c, s, n: _resize_crops(c, s, n, ops.LINEAR), 4),
    "resize crops packed": (lambda c, s, n: _resize_crops(c, s, n, ops.LINEAR, packed=True), 6),
    "chain crops": (lambda c, s, n: _resize_crops(c, s, n, ops.LINEAR, chain=True), 8),
    "nearest crops": (lambda c, s, n: _resize_crops(c, s, n, ops.NEAREST), 4),
    "triangular crops": (lambda c, s, n: _resize_crops(c, s, n, ops.TRIANGULAR), 4),  # (in batch order)
    "triangular crops sorted": (lambda c, s, n: _resize_crops(c, s, n, ops.TRIANGULAR, o=24), 5),
    "crop": (_crop, 2),
    "flip": (_flip, 2),
    "twist": (_twist, 4),
    "twist windows": (lambda c, s, n: _twist(c, s, n, True), 6),
    "brightness": (_brightness, 1),
    "rotate": (_rotate, 6),
    "rotate windows": (lambda c, s, n: _rotate(c, s, n, True), 8),
}


@pytest.mark.parametrize("what", sorted(MAKERS))
@pytest.mark.parametrize("size", ["one", "few", "full", "over"])
def test_records_and_table_agree(ctx, ctx_table, what, size):
    import torch
    make, words = MAKERS[what]
    n = {"one": 1, "few": 19, "full": 768 // words, "over": 768 // words + 1}[size]
    got = []
    for c in (ctx, ctx_table):
        op, img = make(c, 17 + n, n)
        route = "rows=table" if c is ctx_table or size == "over" else "rows=arguments" if size in ("one", "few") else "rows=arguments words=%d" % words
        assert route in op.plan, op.plan
        out = op.alloc_output(fill=3)
        src = torch.from_numpy(img).cuda()
        op.launch(src, out)
        op.launch(src, out)  # (the rows of one update serve any number of launches)
        c.sync()
        got.append(out.cpu().numpy())
    assert np.array_equal(got[0].view(np.uint8), got[1].view(np.uint8))


def test_updates_in_flight_keep_their_own_rows(ctx):
    """Twelve updates and launches without a wait, records and table in turn (the packed layout's 192 samples fit, 193 do not):
    every output has the rows of its own update."""
    import torch
    n, h, w = 193, 20, 32
    rng = np.random.default_rng(4)
    img = rng.integers(0, 256, (n, h, w, 3), dtype=np.uint8)
    src = torch.from_numpy(img).cuda()
    sd = ops.desc(n, h, w, ops.NHWC, ops.UINT8)
    op = ops.ColorTwist(ctx, sd, sd)
    roi = np.tile(np.array([0, 0, w, h], np.uint32), (n, 1))
    outs, args = [], []
    for i in range(12):
        f = lambda lo, hi: rng.uniform(lo, hi, n).astype(np.float32)  # noqa: E731
        hue = f(-30, 30) if i % 2 else np.full(n, 11.0, np.float32)  # (three factors a sample: 579 dwords; four: 772)
        args.append((f(0.5, 1.5), f(-9, 9), hue, f(0.5, 1.5)))
        op.update(roi, *args[-1])
        outs.append(op.alloc_output())
        op.launch(src, outs[-1])
    ctx.sync()
    for a, out in zip(args, outs):
        assert np.array_equal(out.cpu().numpy(), orc.color_twist(img, roi, *a))


def test_coordinates_beyond_a_record(ctx):
    """A window that starts behind column 16383 takes the table."""
    import torch
    rng = np.random.default_rng(5)
    img = rng.integers(0, 256, (2, 4, 16600, 3), dtype=np.uint8)
    roi = np.array([[16500, 0, 96, 4], [3, 0, 96, 4]], np.uint32)
    d = np.array([48, 48], np.uint32), np.array([4, 4], np.uint32)
    op = ops.Resize(ctx, ops.desc(2, 4, 16600, ops.NHWC, ops.UINT8), ops.desc(2, 4, 48, ops.NHWC, ops.UINT8), ops.LINEAR)
    op.update(roi, *d)
    assert "rows=table" in op.plan, op.plan
    out = op.alloc_output()
    op.launch(torch.from_numpy(img).cuda(), out)
    ctx.sync()
    assert np.array_equal(out.cpu().numpy(), orc.resize(img, roi, *d, 4, 48, interp=orc.LINEAR))


@pytest.mark.parametrize("width", [16383, 16384])
@pytest.mark.parametrize("interp", [ops.LINEAR, ops.NEAREST, ops.TRIANGULAR])
def test_widest_resized_image_of_a_record(ctx, width, interp):
    """Ratios are made from the sizes up to 14 bits of either; a wider resized image takes the table."""
    import torch
    rng = np.random.default_rng(6)
    n, h, w, o = 3, 5, 16390, 40
    img = rng.integers(0, 256, (n, h, w, 3), dtype=np.uint8)
    roi = np.array([[0, 0, 16383, 5], [7, 1, 16001, 3], [5000, 0, 9000, 5]], np.uint32)
    dw, dh = np.full(n, width, np.uint32), np.full(n, 4, np.uint32)
    crop = np.array([[0, 0, o, 4], [16300, 1, o, 3], [8001, 0, o - 3, 4]], np.uint32)
    scale, bias = orc.cmn_scale_bias(wl.MEAN, wl.STD, n)
    op = ops.Resize(ctx, ops.desc(n, h, w, ops.NHWC, ops.UINT8), ops.desc(n, 4, o, ops.NCHW, ops.FP32), interp)
    op.update_cmn(roi, dw, dh, scale, bias, crop_roi=crop)
    assert ("rows=arguments" if width == 16383 else "rows=table") in op.plan, op.plan
    out = op.alloc_output()
    op.launch(torch.from_numpy(img).cuda(), out)
    ctx.sync()
    got = out.cpu().numpy()
    exp = orc.resize(img, roi, dw, dh, 4, width, interp=interp, scale=scale, bias=bias, layout=ops.NCHW, dtype=ops.FP32)
    for i, (x, y, cw, ch) in enumerate(crop.astype(int)):
        assert np.array_equal(got[i, :, :ch, :cw].view(np.uint32), exp[i, :, y:y + ch, x:x + cw].view(np.uint32)), i
