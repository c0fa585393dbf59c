"""Warps to interleaved bytes whose rows leave by tiles and by teams of four tiles, bit for bit against the oracle: widths around tiles (32) and
teams (128), heights that end inside a tile, samples smaller than the tensor (the padding stays untouched), destinations off 16 and 128
bytes, tiles outside the window beside tiles inside it, boxes too large for LDS in the same workgroup."""
import numpy as np
import pytest

from oracle import orc
from rocal_amd import ops, workloads as wl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx_together():
    """(rows leave together in large batches only, unless told)"""
    from conftest import _ctx_with_env
    c = _ctx_with_env(RMX_TUNE_WARP_TOGETHER=2)
    yield c
    c.close()


@pytest.mark.parametrize("interp", [ops.LINEAR, ops.NEAREST])
@pytest.mark.parametrize("W,H,off", [(128, 64, 0), (256, 70, 0), (256, 33, 16), (256, 33, 1), (128, 31, 3), (127, 40, 0), (272, 50, 0), (304, 45, 0), (97, 64, 0), (400, 90, 0), (32, 32, 0), (31, 20, 0)])
def test_rows_of_tiles_and_teams(ctx_together, interp, W, H, off):
    import torch
    ctx = ctx_together
    rng = np.random.default_rng(W * 7 + H + off)
    n = 5
    img = wl.smooth_noise(rng, n, H, W, sigma=1.0)
    roi = np.tile(np.array([0, 0, W, H], np.uint32), (n, 1))
    roi[2] = (W // 4, H // 3, W // 2, H // 2)
    affine = np.array([[1, 0, 0, 1, 0, 0], [0.9, 0.25, -0.2, 1.1, 3.5, -2.25], [1, 0, 0, 1, 0.5, 0.25], [0.7, -0.7, 0.7, 0.7, 9.0, 2.0],
                       [6.0, 0.5, -0.5, 6.0, 0.0, 0.0]], np.float32)
    dw = np.array([W, W, W, max(W - 5, 1), W], np.uint32)
    dh = np.array([H, H, max(H - 7, 1), H, H], np.uint32)
    exp = orc.warp_affine(img, roi, np.stack([orc.affine_from_rocal(a) for a in affine]), dw, dh, H, W, interp=interp)
    sd = ops.desc(n, H, W, ops.NHWC, ops.UINT8)
    op = ops.WarpAffine(ctx, sd, sd, interp)
    op.update(roi, affine, dw, dh)
    buf = torch.full((n * H * W * 3 + 256,), 9, dtype=torch.uint8, device="cuda")
    out = buf[off:off + n * H * W * 3].view(n, H, W, 3)
    op.launch(torch.from_numpy(img).cuda(), out)
    ctx.sync()
    got, want = out.cpu().numpy(), np.full((n, H, W, 3), 9, np.uint8)
    for i in range(n):
        want[i, :dh[i], :dw[i]] = exp[i, :dh[i], :dw[i]]
    assert np.array_equal(got, want), "%d values differ (%s)" % (int((got != want).sum()), op.plan)
    # (four tiles side by side that are whole cache lines; the nearest pixel's tiles at any place, bilinear ones at multiples of 16 bytes)
    mode = "teams" if W % 128 == 0 else "tiles" if interp == ops.NEAREST or W % 16 == 0 else "lanes"
    assert "leave=%s" % mode in op.plan, op.plan
    assert op.kernel_name == ("rmx_warp_kernel" if mode == "lanes" else "rmx_warp_rows_kernel") + ("(raw)" if W % 4 == 0 else ""), op.kernel_name
    rest = buf.cpu().numpy()
    assert (rest[:off] == 9).all() and (rest[off + n * H * W * 3:] == 9).all()


@pytest.mark.parametrize("interp", [ops.LINEAR, ops.NEAREST])
@pytest.mark.parametrize("W,mode", [(256, "teams"), (272, "tiles")])
def test_sources_at_any_phase(ctx_together, interp, W, mode):
    """Packed images of odd widths (rows at every byte phase) to teams and tiles, the last one ending on the buffer's last byte."""
    import torch
    ctx = ctx_together
    rng = np.random.default_rng(W)
    widths, heights = np.array([131, 201, 77, 255], np.uint32), np.array([70, 33, 64, 50], np.uint32)
    n, SH, SW, H = len(widths), 70, 255, 66
    img = np.zeros((n, SH, SW, 3), np.uint8)
    parts = []
    for i in range(n):
        img[i, :heights[i], :widths[i]] = rng.integers(0, 256, (int(heights[i]), int(widths[i]), 3), dtype=np.uint8)
        parts.append(img[i, :heights[i], :widths[i]].reshape(-1))
    sizes = np.array([p.size for p in parts], np.int64)
    offsets = (np.cumsum(sizes) - sizes).astype(np.uint64)
    src = np.concatenate(parts)
    roi = np.stack([np.zeros(n), np.zeros(n), widths, heights], 1).astype(np.uint32)
    affine = np.array([[1, 0, 0, 1, 0, 0], [0.9, 0.25, -0.2, 1.1, 3.5, -2.25], [0.3, 0.0, 0.0, 1.0, 0.5, 0.25], [0.9, -0.4, 0.4, 0.9, 9.0, 2.0]], np.float32)
    dw, dh = np.array([W, W, W - 5, W], np.uint32), np.array([H, 33, H, 61], np.uint32)
    exp = orc.warp_affine(img, roi, np.stack([orc.affine_from_rocal(a) for a in affine]), dw, dh, H, W, interp=interp)
    op = ops.WarpAffine(ctx, ops.desc(n, SH, SW, ops.NHWC, ops.UINT8), ops.desc(n, H, W, ops.NHWC, ops.UINT8), interp)
    op.set_ragged_source(offsets, widths, heights, src.size)
    op.update(roi, affine, dw, dh)
    assert op.kernel_name == "rmx_warp_rows_kernel" and "leave=%s" % mode in op.plan, (op.kernel_name, op.plan)
    out = op.alloc_output(fill=9)
    op.launch(torch.from_numpy(src).cuda(), out)
    ctx.sync()
    got, want = out.cpu().numpy(), np.full((n, H, W, 3), 9, np.uint8)
    for i in range(n):
        want[i, :dh[i], :dw[i]] = exp[i, :dh[i], :dw[i]]
    assert np.array_equal(got, want), "%d values differ (%s)" % (int((got != want).sum()), op.plan)
