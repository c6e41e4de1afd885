"""The polar remaps' 32x8 and the tape warp's 64x4 tiles at sizes that no tile
divides, from the smallest each call takes, against the oracle, byte for byte."""
import numpy as np
import pytest

from helpers import rand_img
from oracles import P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(4, 4), (30, 6), (34, 10), (62, 18), (96, 64), (1366, 766)])
def test_polar(ctx, orc, W, H):
    src, dst = rand_img(W, W * H), rand_img(H, W * H)
    m0, m1 = np.zeros(W * H * 2, np.int32), np.zeros(W * H * 2, np.int32)
    orc.orc_polar_maps(P(m0), P(m1), W, H, W, H)
    ctx.polar_create(W, H)
    s, d = ctx.upload(src), ctx.empty(W * H)
    for inverse, m in ((0, m0), (1, m1)):
        want = np.zeros(W * H, np.uint32)
        orc.orc_polar_blit(P(want), P(src), P(m), W, H, W, 8)
        ctx.polar_blit(d, s, W, H, inverse)
        assert np.array_equal(d.numpy(), want), inverse
        a, want = ctx.upload(dst), dst.copy()
        orc.orc_polar_blit_a(P(want), P(src), P(m), W, H, W, 8)
        ctx.polar_blit_a(a, s, W, H, inverse)
        assert np.array_equal(a.numpy(), want), inverse


@pytest.mark.parametrize("W,H", [(2, 2), (3, 5), (63, 3), (65, 9), (129, 66), (1367, 767)])
def test_tape_warp(ctx, orc, W, H):
    lut = np.zeros(2049, np.float32)
    orc.orc_cos_lut(P(lut))
    src = rand_img(7 * W + H, W * H)
    s, d = ctx.upload(src), ctx.empty(W * H)
    for strength, speed in ((6.5, 0.02), (-300.0, 0.7)):
        want = np.zeros(W * H, np.uint32)
        orc.orc_tape_warp32(P(want), P(src), W, H, strength, speed, P(lut))
        ctx.tape_warp32(d, s, W, H, strength, speed)
        assert np.array_equal(d.numpy(), want), (strength, speed)
