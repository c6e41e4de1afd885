"""The ball's wave per row (k_ball): ray lengths about the 64 steps a wave takes
at once, whose texels are read a chunk ahead, and the beams' alpha ramp over
short and long remainders of a row, whose chunks are products inside a binade
and sums across one.  Byte for byte against the oracle."""
import numpy as np
import pytest

from cookiedough_amd import workloads as wl
from oracles import P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(1280, 720), (2048, 64), (68, 24)])
def test_ray_lengths_and_remainders(ctx, orc, W, H):
    bm = wl.ball_maps(W, H)
    m0, m1 = np.zeros(2 * W * H, np.int32), np.zeros(2 * W * H, np.int32)
    orc.orc_polar_maps(P(m0), P(m1), W, H, W, H)
    ctx.ball_create(bm, W, H)
    tgt, d = ctx.empty(W * H), ctx.empty(W * H)
    for k, (ray, radius) in enumerate([(1, 30.0), (63, 20.0), (64, 35.0), (65, 10.0), (128, 3.0), (512, 40.0),
                                       (1023, 25.0), (1024, 40.0)]):
        for beams in (0.0, 1.0):
            prm = wl.ball_frames(1, int(beams), t0=3.0 + k)[0]
            prm.rayLength, prm.radius, prm.hasBeams, prm.blur = float(ray), radius, beams, 0.0
            print("ball", W, H, ray, radius, beams, flush=True)
            host_t = np.full(W * H, 0x01020304, np.uint32)
            ctx.memset32(tgt, 0x01020304, W * H)
            ctx.ball_draw(d, tgt, W, H, [prm])
            ctx.sync()
            want = np.zeros(W * H, np.uint32)
            assert orc.orc_ball_draw(P(want), P(host_t), W, H, P(bm["heightMaps"]), P(bm["colorMaps"]),
                                     P(bm["beamMaps"]), P(bm["envMap"]), P(bm["backgrounds"]), P(bm["halo"]),
                                     P(m0), P(prm.as_array()), 8) == 0
            assert np.array_equal(d.numpy(), want), (ray, beams)
            assert np.array_equal(tgt.numpy(), host_t), (ray, beams)
