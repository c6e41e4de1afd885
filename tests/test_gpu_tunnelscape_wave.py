"""The tunnelscape's wave per row (code/tunnelscape.cpp:44-100) against the
oracle at the edges of its range, and the integer form of its height (one
division for the reference's FP32 quotient and its integer division) against
the reference's steps for every map height and step."""
import numpy as np
import pytest

from cookiedough_amd import workloads as wl
from oracles import P

MOVES = [(0.3, 1.2, 2.0, 0.0), (-0.7, -0.9, 1.0, 3.5), (0.0, 0.004, 0.5, 1.0)]


# heights are at least 120: rows up to 120 pixels draw nothing, 121 the least
@pytest.mark.gpu
@pytest.mark.parametrize("W,H", [(8, 8), (120, 9), (121, 33), (1366, 65), (4096, 17), (64, 4096)])
def test_rows_equal_oracle(ctx, orc, W, H):
    m = wl.tunnelscape_maps(1)
    ctx.tunnelscape_create(m.height, m.color, m.fog)
    d = ctx.empty(W * H)
    for su, sv, sp, t in MOVES:
        ctx.memset32(d, 0x5a5a5a5a, W * H)
        ctx.tunnelscape_rows(d, W, H, su, sv, sp, t)
        ref = np.zeros(W * H, np.uint32)
        orc.orc_tscape_frame(P(ref), W, H, P(m.height), P(m.color), P(m.fog), su, sv, sp, t, 8)
        assert np.array_equal(d.numpy(), ref), (W, H, su, sv)


def test_height_form():
    f32 = np.float32
    h = np.arange(160)[:, None]
    n = np.arange(1, 513)[None, :]
    scale = f32(f32(720) / f32(1280)) * f32(0.5)
    ref = (((255 - h - 96) << 8).astype(f32) / scale).astype(np.int64) // n * 160 // 256 + 120
    num, den = ((159 - h) << 13).astype(f32), (9 * n).astype(f32)
    near = (f32(1) / den).astype(f32)
    for rcp in (near, np.nextafter(near, f32(0)), np.nextafter(near, f32(1))):
        q = np.trunc((num.astype(np.float64) * rcp.astype(np.float64) - 0.5).astype(f32)).astype(np.int64)
        q += num.astype(np.int64) - q * den.astype(np.int64) >= den
        assert np.array_equal((q * 160 >> 8) + 120, ref)
