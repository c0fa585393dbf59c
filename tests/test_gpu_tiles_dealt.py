"""Resizes whose x-tiles are dealt to several wavefronts (small batches): the same bits as with one wavefront per window, and as the oracle.
Widths at the edges of tiles and of groups, samples of one tile beside samples of many (whose other wavefronts have nothing to do),
mirrors, windows up to the last byte of the buffer."""
import numpy as np
import pytest

from oracle import orc
from rocal_amd import ops, workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout,dtype", [(ops.NCHW, ops.FP16), (ops.NHWC, ops.FP16), (ops.NCHW, ops.FP32), (ops.NHWC, ops.FP32), (ops.NHWC, ops.UINT8)])
@pytest.mark.parametrize("W,OW,interp", [(700, 256, ops.LINEAR), (701, 299, ops.LINEAR), (700, 263, ops.LINEAR), (501, 131, ops.LINEAR), (701, 513, ops.NEAREST)])
def test_tiles_of_a_window_in_several_wavefronts(layout, dtype, W, OW, interp):
    import torch
    from conftest import _ctx_with_env
    rng = np.random.default_rng(W + OW + dtype)
    n, H, OH = 3, 90, 23
    img = wl.smooth_noise(rng, n, H, W, sigma=1.0)
    roi = np.array([[0, 0, W, H], [3, 1, W - 3, H - 1], [W - 60, H - 30, 60, 30]], np.uint32)
    dw, dh = np.array([OW, OW - 8, 40], np.uint32), np.array([OH, OH - 1, 9], np.uint32)
    mirror = np.array([0, 1, 1], np.uint32)
    norm = dtype != ops.UINT8
    s, b = orc.cmn_scale_bias(wl.MEAN, wl.STD, n)
    kw = dict(scale=s if norm else None, bias=b if norm else None)
    exp = orc.resize(img, roi, dw, dh, OH, OW, interp=interp, mirror=mirror, layout=layout, dtype=dtype, **kw)
    src = torch.from_numpy(img.reshape(-1).copy()).cuda().view(n, H, W, 3)
    got = []
    for split in (0, 1):
        c = _ctx_with_env(RMX_TUNE_DMA_SPLIT=split)
        op = ops.Resize(c, ops.desc(n, H, W, ops.NHWC, ops.UINT8), ops.desc(n, OH, OW, layout, dtype), interp)
        if norm:
            op.update_cmn(roi, dw, dh, s, b, mirror)
        else:
            op.update(roi, dw, dh, mirror)
        assert (op.kernel_name == "rmx_resize_split_kernel") == bool(split) == ("split=" in op.plan), (op.kernel_name, op.plan)
        waves = int(op.plan.split("waves=")[1].split()[0])
        assert waves == n * 6 if not split else waves > n * 6, op.plan
        out = op.alloc_output(fill=3)
        op.launch(src, out)
        c.sync()
        got.append(out.cpu().numpy())
        c.close()
    assert np.array_equal(got[0].view(np.uint8), got[1].view(np.uint8))
    for i in range(n):
        g, e = (got[1][i][:, :dh[i], :dw[i]], exp[i][:, :dh[i], :dw[i]]) if layout == ops.NCHW else (got[1][i][:dh[i], :dw[i]], exp[i][:dh[i], :dw[i]])
        assert np.array_equal(np.ascontiguousarray(g).view(np.uint8), np.ascontiguousarray(e).view(np.uint8)), (i, op.plan)


@pytest.mark.parametrize("n,tiles,parts", [(27, 1, 1), (27, 2, 2), (5, 1, 2), (5, 2, 2)])
def test_batches_of_mostly_one_tile(ctx, n, tiles, parts):
    """Windows of one tile beside one window of two: dealt in small batches only, where their idle wavefronts cost less than the wait for the
    second tile; whole batches of two tiles in larger ones too."""
    import torch
    rng = np.random.default_rng(n)
    H, W, OH, OW = 300, 700, 266, 249
    img = rng.integers(0, 256, (n, H, W, 3), dtype=np.uint8)
    roi = np.tile(np.array([[0, 0, 200 if tiles == 1 else W, 200]], np.uint32), (n, 1))
    roi[n - 1, 2] = W
    dw, dh = np.full(n, OW, np.uint32), np.full(n, OH, np.uint32)
    s, b = orc.cmn_scale_bias(wl.MEAN, wl.STD, n)
    op = ops.Resize(ctx, ops.desc(n, H, W, ops.NHWC, ops.UINT8), ops.desc(n, OH, OW, ops.NCHW, ops.FP16), ops.LINEAR, flags=ops.F_QUANTIZE_U8)
    op.update_cmn(roi, dw, dh, s, b, None)
    assert int(op.plan.split("waves=")[1].split()[0]) == n * 67 * parts, op.plan
    out = op.alloc_output()
    op.launch(torch.from_numpy(img).cuda(), out)
    ctx.sync()
    exp = orc.resize(img, roi, dw, dh, OH, OW, interp=orc.LINEAR, scale=s, bias=b, layout=orc.NCHW, dtype=orc.FP16, flags=orc.F_QUANTIZE_U8)
    assert np.array_equal(out.cpu().numpy().view(np.uint8), exp.view(np.uint8)), op.plan


@pytest.mark.parametrize("layout,dtype", [(ops.NCHW, ops.FP16), (ops.NHWC, ops.FP16), (ops.NCHW, ops.FP32), (ops.NHWC, ops.FP32)])
@pytest.mark.parametrize("chain", ["none", "linear", "twist"])
@pytest.mark.parametrize("OW", [264, 261])
def test_quantised_chains_in_several_wavefronts(layout, dtype, chain, OW):
    """Resize, colour node, normalisation in one launch (each wavefront of a window has the colour tables of its own): the same bits as with one
    wavefront per window, which the chain's own tests hold against the nodes one by one."""
    import torch
    from conftest import _ctx_with_env
    rng = np.random.default_rng(OW + dtype + layout)
    n, H, W, OH = 3, 90, 701, 22
    img = wl.smooth_noise(rng, n, H, W, sigma=1.0)
    roi = np.array([[0, 0, W, H], [3, 1, W - 3, H - 1], [W - 60, H - 30, 60, 30]], np.uint32)
    dw, dh = np.array([OW, OW - 8, 40], np.uint32), np.array([OH, OH - 1, 9], np.uint32)
    mirror = np.array([0, 1, 1], np.uint32)
    s, b = orc.cmn_scale_bias(wl.MEAN, wl.STD, n)
    flag = {"none": 0, "linear": ops.F_COLOR_LINEAR, "twist": ops.F_COLOR_TWIST}[chain]
    u = lambda lo, hi: rng.uniform(lo, hi, n).astype(np.float32)  # noqa: E731
    colour = {"none": None, "linear": (u(0.6, 1.4), u(-20, 20), u(100, 150)), "twist": (u(0.6, 1.4), u(-20, 20), u(-18, 200), u(0.6, 1.4))}[chain]
    src = torch.from_numpy(img).cuda()
    got = []
    for split in (0, 1):
        c = _ctx_with_env(RMX_TUNE_DMA_SPLIT=split)
        op = ops.Resize(c, ops.desc(n, H, W, ops.NHWC, ops.UINT8), ops.desc(n, OH, OW, layout, dtype), ops.LINEAR, flags=ops.F_QUANTIZE_U8 | flag)
        if colour is None:
            op.update_cmn(roi, dw, dh, s, b, mirror)
        else:
            op.update_color_cmn(roi, dw, dh, s, b, colour, mirror)
        assert (op.kernel_name == "rmx_resize_split_kernel") == bool(split), (op.kernel_name, op.plan)
        out = op.alloc_output(fill=3)
        op.launch(src, out)
        c.sync()
        got.append(out.cpu().numpy())
        c.close()
    assert np.array_equal(got[0].view(np.uint8), got[1].view(np.uint8))
    if colour is None:
        exp = orc.resize(img, roi, dw, dh, OH, OW, interp=orc.LINEAR, mirror=mirror, layout=layout, dtype=dtype, scale=s, bias=b, flags=orc.F_QUANTIZE_U8)
        for i in range(n):
            x = (i, slice(None), slice(0, dh[i]), slice(0, dw[i])) if layout == ops.NCHW else (i, slice(0, dh[i]), slice(0, dw[i]))
            assert np.array_equal(np.ascontiguousarray(got[1][x]).view(np.uint8), np.ascontiguousarray(exp[x]).view(np.uint8)), i
