"""Parameter rows that go through the ring of table slots: more updates and launches in flight than the ring has slots, rows in the
arguments and in the table by turns, and a captured launch that reads a table slot."""
import numpy as np
import pytest

from oracle import orc
from rocal_amd import ops

pytestmark = pytest.mark.gpu
N, H, W = 9, 20, 32


def _context(stream="torch", **env):
    with pytest.MonkeyPatch.context() as m:
        for k, v in env.items():
            m.setenv(k, str(v))
        return ops.Context(0, stream=stream)


def _twist_args(rng):
    f = lambda lo, hi: rng.uniform(lo, hi, N).astype(np.float32)  # noqa: E731
    return f(0.5, 1.5), f(-9, 9), f(-30, 30), f(0.5, 1.5)


def test_more_updates_in_flight_than_slots():
    import torch
    c = _context(RMX_TUNE_COMPACT=0)
    rng = np.random.default_rng(41)
    img = rng.integers(0, 256, (N, H, W, 3), dtype=np.uint8)
    src = torch.from_numpy(img).cuda()
    sd = ops.desc(N, H, W, ops.NHWC, ops.UINT8)
    roi = np.tile(np.array([0, 0, W, H], np.uint32), (N, 1))
    op = ops.ColorTwist(c, sd, sd)
    outs = [op.alloc_output() for _ in range(37)]  # (four times round the ring and into its second half)
    args = [_twist_args(rng) for _ in outs]
    for a, out in zip(args, outs):
        op.update(roi, *a)
        assert "rows=table" in op.plan, op.plan
        op.launch(src, out)
    c.sync()
    for k, (a, out) in enumerate(zip(args, outs)):
        assert np.array_equal(out.cpu().numpy(), orc.color_twist(img, roi, *a)), k


@pytest.mark.parametrize("table", [True, False])
def test_a_captured_launch_keeps_its_rows(table):
    """The launch is recorded behind several updates; other ops of the context fill and read their own slots between the replays."""
    import torch
    from rocal_amd._lib import RmxError
    s = torch.cuda.Stream()
    c = _context(s.cuda_stream, RMX_TUNE_COMPACT=int(not table))
    rng = np.random.default_rng(42)
    sd = ops.desc(N, H, W, ops.NHWC, ops.UINT8)
    roi = np.tile(np.array([0, 0, W, H], np.uint32), (N, 1))
    op, other = ops.ColorTwist(c, sd, sd), ops.ColorTwist(c, sd, sd)
    for _ in range(6):
        keep = _twist_args(rng)
        op.update(roi, *keep)
    assert ("rows=table" if table else "rows=arguments") in op.plan, op.plan
    with torch.cuda.stream(s):
        src = torch.zeros((N, H, W, 3), dtype=torch.uint8, device="cuda")
        out, out2 = op.alloc_output(), other.alloc_output()
        op.launch(src, out)
        s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        op.launch(src, out)
    for rep in range(10):
        img = rng.integers(0, 256, (N, H, W, 3), dtype=np.uint8)
        args = _twist_args(rng)
        with pytest.raises(RmxError, match="recorded into a HIP graph"):
            op.update(roi, *args)
        other.update(roi, *args)
        with torch.cuda.stream(s):
            src.copy_(torch.from_numpy(img))
            other.launch(src, out2)
            out.zero_()
            g.replay()
            s.synchronize()
        assert np.array_equal(out.cpu().numpy(), orc.color_twist(img, roi, *keep)), rep
        assert np.array_equal(out2.cpu().numpy(), orc.color_twist(img, roi, *args)), rep
