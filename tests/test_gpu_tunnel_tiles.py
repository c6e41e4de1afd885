"""The tunnel's vertical pass in LDS tiles (k_tunnel_v_tile), which launches of
up to 4096 tiles (fewer of short segments) with segments up to 64 rows take while
segment and window fit 254 rows of LDS: both sides of each of these limits, segments that rows do not
divide, columns that tiles do not, windows clipped at either end and at both,
and a batch of jobs with different windows.  Bit for bit against the oracle."""
import contextlib

import numpy as np
import pytest

from cookiedough_amd import workloads as wl
from cookiedough_amd._lib import CKD_FX_TUNNEL, CKD_SHADE_FP32
from oracles import P

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def _segment(ctx, rows):
    saved, t = ctx.get_tuning(), ctx.get_tuning()
    t.tunnelVSeg = rows
    ctx.set_tuning(t)
    try:
        yield
    finally:
        ctx.set_tuning(saved)


def _want(orc, W, H, grid, tex, r):
    ref, o0, o1 = (np.zeros(W * H, np.uint32) for _ in range(3))
    orc.orc_tunnel_frame(P(ref), P(o0), P(o1), W, H, P(grid), P(tex), 9, r, 8)
    return ref


@pytest.mark.parametrize("W,H,r,seg", [
    (256, 255, 111, 32), (256, 255, 112, 32), (200, 257, 95, 64), (200, 257, 96, 64),   # 254 rows and more
    (130, 131, 12, 64), (130, 131, 12, 65), (333, 77, 33, 8), (321, 100, 1, 9),         # 64 rows and more
    (1280, 1632, 3, 8), (1280, 1640, 3, 8),                                             # 4080 and 4100 tiles
    (65, 65, 32, 32), (127, 129, 32, 63), (64, 33, 16, 32)])
def test_frame(ctx, orc, W, H, r, seg):
    tex, grid = wl.noise_texture(0, 9), wl.tunnel_grid(W, H, 3.0 + r)
    d, tmp = ctx.empty(W * H), ctx.empty(W * H)
    with _segment(ctx, seg):
        ctx.tunnel_frame(d, tmp, W, H, ctx.upload(grid), ctx.upload(tex), 9, r)
        got = d.numpy()
    assert np.array_equal(got, _want(orc, W, H, grid, tex, r))


# short segments give way to the ring from 1500 tiles on (at 16 rows only below
# radius 8), the others from 4096 on; past the ring from 860000 rows read on
@pytest.mark.parametrize("W,H,r,seg", [
    (1280, 600, 3, 8), (1280, 601, 3, 8), (1280, 1216, 7, 16), (1280, 1216, 8, 16), (1280, 1216, 7, 24),
    (4096, 2112, 2, 33), (4096, 2113, 2, 33), (1280, 1600, 103, 8), (1280, 1608, 103, 8)])
def test_limits(ctx, orc, W, H, r, seg):
    test_frame(ctx, orc, W, H, r, seg)


@pytest.mark.parametrize("seg", [16, 32, 64])
def test_batch_of_windows(ctx, orc, seg):
    tex = wl.noise_texture(0, 9)
    shapes = [(320, 180, 1), (640, 360, 32), (328, 200, 64), (96, 64, 7)]
    total = sum(w * h for w, h, _ in shapes)
    out, tmp, at, reqs, grids, held = ctx.empty(total), ctx.empty(total), 0, [], [], []
    for w, h, r in shapes:
        grids.append(wl.tunnel_grid(w, h, 1.0 + r))
        held.append(ctx.upload(grids[-1]))
        reqs.append(wl.make_request(wl.BatchItem(CKD_FX_TUNNEL, w, h, 0.0, r), out.ptr + 4 * at, None, None,
                                    held[-1].ptr))
        at += w * h
    with _segment(ctx, seg):
        ctx.render_batch(reqs, None, CKD_SHADE_FP32, ctx.upload(tex), 9, tmp, total)
        got = out.numpy()
    at = 0
    for (w, h, r), grid in zip(shapes, grids):
        assert np.array_equal(got[at:at + w * h], _want(orc, w, h, grid, tex, r)), (w, h, r)
        at += w * h
