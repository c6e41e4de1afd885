"""The SDF tracer of one frame (k_sdf): a 16x16 tile keeps the spheres that can
be its rays' nearest surface and evaluates them on the stretch of the rays that
can be near any.  Both leave the full minimum, so frames equal the FP64 render
as they do without: sizes no tile divides, tiles wider than the cull allows
(a wide lens over few pixels), cameras below the ground, among the spheres and
far from the origin, crowds, negative radii, and marches that end below a
surface."""
import numpy as np
import pytest

from cookiedough_amd import workloads as wl
from cookiedough_amd._lib import CKD_SHADE_FP16, CKD_SHADE_FP32
from helpers import sdf_fp64, sdf_report

pytestmark = pytest.mark.gpu


def _check(ctx, orc, sc, W, H, t, shading=CKD_SHADE_FP32):
    out = ctx.empty(W * H)
    ctx.sdf_render(out, W, H, sc, wl.sdf_camera(sc, t), shading)
    got = out.numpy()
    ctx.free(out)
    ref, _, cond = sdf_fp64(orc, sc, W, H, t)
    es = sdf_report(got, ref, cond)
    print("sdf", W, H, sc.nSpheres, es, flush=True)
    assert es["max_outside_rounding_decided"] <= 2, es


@pytest.mark.parametrize("n", [1, 8, 32])
@pytest.mark.parametrize("W,H", [(1, 1), (17, 33), (641, 363), (9, 501)])
def test_sizes(ctx, orc, W, H, n):
    _check(ctx, orc, wl.sdf_scene(3, n, 64), W, H, 4.2)


@pytest.mark.parametrize("W,H,n", [(640, 400, 6), (640, 400, 7), (800, 532, 6), (832, 536, 6), (640, 400, 16),
                                   (640, 400, 17), (960, 540, 11), (960, 540, 12), (64, 64, 0)])
def test_either_side_of_the_forms(ctx, orc, W, H, n):
    """few spheres and few tiles; tiles that keep all spheres; tiles that cull"""
    sc = wl.sdf_scene(3, max(n, 1), 64)
    sc.nSpheres = n
    _check(ctx, orc, sc, W, H, 4.2)


@pytest.mark.parametrize("height", [-4.5, 0.0, 30.0])
@pytest.mark.parametrize("radius", [0.5, 4.0, 40.0])
def test_cameras_anywhere(ctx, orc, height, radius):
    sc = wl.sdf_scene(5, 8, 64)
    sc.camHeight, sc.camRadius = height, radius
    _check(ctx, orc, sc, 320, 200, 1.0)


@pytest.mark.parametrize("focal", [0.02, 0.3, 4.0])
def test_lenses(ctx, orc, focal):
    sc = wl.sdf_scene(6, 8, 64)
    sc.focal = focal
    _check(ctx, orc, sc, 96, 10, 2.0)
    _check(ctx, orc, sc, 200, 120, 2.0)


@pytest.mark.parametrize("eps", [1e-3, -0.05])
def test_crowd_with_holes(ctx, orc, eps):
    sc = wl.sdf_scene(11, 32, 96)
    geo = wl.Rng(4, 77).uniform(4 * 32).reshape(32, 4)
    for i in range(32):
        for k in range(3):
            sc.sphere[i][k] = 1.6 * (2.0 * geo[i, k] - 1.0)
        sc.sphere[i][3] = (0.15 + 0.2 * geo[i, 3]) * (-1.0 if i % 8 == 3 else 1.0)
    sc.eps = eps
    _check(ctx, orc, sc, 331, 187, 2.5)


@pytest.mark.parametrize("shading", [CKD_SHADE_FP32, CKD_SHADE_FP16])
@pytest.mark.parametrize("W,H", [(200, 120), (1000, 600)])
def test_every_length_of_a_list(ctx, orc, W, H, shading):
    """lists of whole groups of four spheres and every remainder, kept whole (the
    small frame) and culled"""
    for n in range(33):
        sc = wl.sdf_scene(n, max(n, 1), 64)
        sc.nSpheres = n
        _check(ctx, orc, sc, W, H, 4.2, shading)
