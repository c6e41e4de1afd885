"""The batched SDF tracer's chunks (k_sdf_persistent): their side follows the
batch's pixels (8 up to 2 M and 8 spheres, 16 up to 32 M, then 32), they are
traced in 8x8 tiles, and those of 16 and 32 leave out the spheres that can be
the nearest surface to no point of their rays.  None of it may change a byte:
a frame is the same in a batch of every side, also where the camera is below
the ground or inside a sphere, where a chunk needs more than 16 spheres, and
at sizes no tile divides.  Crowded scenes also against the FP64 render."""
import numpy as np
import pytest

from cookiedough_amd import workloads as wl
from cookiedough_amd._lib import CKD_FX_SDF, CKD_SHADE_FP16, CKD_SHADE_FP32
from helpers import sdf_fp64, sdf_report

pytestmark = pytest.mark.gpu

SIDE16, SIDE32 = (2560, 1440, 1), (2560, 1440, 9)  # filler: more than 2 M, more than 32 M pixels


def _frame(ctx, sc, W, H, t, shading, filler=None):
    """the first request of a batch that the filler's requests follow"""
    sizes = [(W, H)] + ([filler[:2]] * filler[2] if filler else [])
    out = ctx.empty(sum(w * h for w, h in sizes))
    reqs, at = [], 0
    for k, (w, h) in enumerate(sizes):
        reqs.append(wl.make_request(wl.BatchItem(CKD_FX_SDF, w, h, t + 0.5 * k), out.ptr + 4 * at, sc, None, None))
        at += w * h
    ctx.memset32(out, 0x12345678, at)
    ctx.render_batch(reqs, sc, shading, None, 9, None, 0)
    got = out.view(0, (W * H,)).numpy()
    ctx.free(out)
    return got


def _crowd(n, seed, half):
    sc = wl.sdf_scene(seed, n, 96)
    geo = wl.Rng(seed, 77).uniform(4 * n).reshape(n, 4)
    for i in range(n):
        for k in range(3):
            sc.sphere[i][k] = half * (2.0 * geo[i, k] - 1.0)
        sc.sphere[i][3] = 0.15 + 0.2 * geo[i, 3]
    return sc


@pytest.mark.parametrize("shading", [CKD_SHADE_FP32, CKD_SHADE_FP16])
@pytest.mark.parametrize("W,H", [(641, 363), (9, 1001), (1279, 15)])
@pytest.mark.parametrize("n", [1, 8])
def test_every_side_gives_the_same_frame(ctx, n, W, H, shading):
    sc = wl.sdf_scene(3, n, 64)
    base = _frame(ctx, sc, W, H, 4.2, shading)
    for filler in (SIDE16, SIDE32):
        assert np.array_equal(_frame(ctx, sc, W, H, 4.2, shading, filler), base), (n, W, H, filler)


@pytest.mark.parametrize("height", [-7.0, -4.5, 0.0, 30.0])
@pytest.mark.parametrize("radius", [0.5, 4.0, 40.0])
def test_cameras_anywhere(ctx, height, radius):
    """below and on the ground, among the spheres, looking straight down"""
    sc = wl.sdf_scene(5, 8, 64)
    sc.camHeight, sc.camRadius = height, radius
    base = _frame(ctx, sc, 320, 200, 1.0, CKD_SHADE_FP32)
    for filler in (SIDE16, SIDE32):
        assert np.array_equal(_frame(ctx, sc, 320, 200, 1.0, CKD_SHADE_FP32, filler), base), filler


@pytest.mark.parametrize("n,half", [(32, 0.8), (32, 2.0), (17, 0.3), (9, 4.0)])
def test_crowded_scenes(ctx, orc, n, half):
    sc = _crowd(n, 11, half)
    W, H, t = 331, 187, 2.5
    a = _frame(ctx, sc, W, H, t, CKD_SHADE_FP32)
    b = _frame(ctx, sc, W, H, t, CKD_SHADE_FP32, SIDE32)
    assert np.array_equal(a, b)
    ref, _, cond = sdf_fp64(orc, sc, W, H, t)
    es = sdf_report(a, ref, cond)
    print("crowd", n, half, es, flush=True)
    assert es["max_outside_rounding_decided"] <= 2, es


def test_graph_replays(ctx):
    """the queues' counters are reset by every replay"""
    sc = wl.sdf_scene(2, 8, 64)
    W, H, n = 640, 360, 20
    out = ctx.empty(n * W * H)
    reqs = ctx.request_array([wl.make_request(wl.BatchItem(CKD_FX_SDF, W, H, 0.3 * k), out.ptr + 4 * k * W * H,
                                              sc, None, None) for k in range(n)])
    ctx.render_batch(reqs, sc, CKD_SHADE_FP16, None, 9, None, 0)
    want = out.numpy()
    g = ctx.batch_graph(reqs, sc, CKD_SHADE_FP16, None, 9, None, 0)
    for _ in range(3):
        ctx.memset32(out, 0, n * W * H)
        g.launch()
        ctx.sync()
        assert np.array_equal(out.numpy(), want)
    g.close()
