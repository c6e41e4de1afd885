"""The 2026 blur's line kernel (k_b26_lines) against the oracle, bit for bit:
lines that fill their waves exactly, by one less and one more, for each number
of pixels a lane takes; few lines and many, one and two a block; several passes a launch,
where two pixels of the next line are carried along, up to as many as there are; spans from none to the longest; both store orders."""
import numpy as np
import pytest

from helpers import rand_img
from oracles import P

pytestmark = pytest.mark.gpu


def _check(ctx, orc, kind, W, H, strength, gain, passes):
    print("blur26", kind, W, H, strength, gain, passes, flush=True)
    n = W * H
    src = np.zeros(n + 4, np.uint32)
    src[:n] = rand_img(W + 3 * H, n)
    want, s0, s1 = (np.zeros(n + 4, np.uint32) for _ in range(3))
    {"h": orc.orc_blur26_h, "v": orc.orc_blur26_v, "2d": orc.orc_blur26}[kind](
        P(want), P(src), W, H, strength, gain, passes, P(s0), P(s1))
    d, s = ctx.empty(n), ctx.upload(src[:n])
    {"h": ctx.blur26_h, "v": ctx.blur26_v, "2d": ctx.blur26}[kind](d, s, W, H, strength, gain, passes)
    got = d.numpy()
    assert np.array_equal(s.numpy(), src[:n])
    ctx.free(s)
    ctx.free(d)
    bad = np.nonzero(got != want[:n])[0]
    assert len(bad) == 0, (len(bad), int(bad[0]) // W, int(bad[0]) % W)


WIDTHS = [4, 5, 191, 192, 193, 319, 320, 321, 448, 449, 576, 577, 639, 641, 960, 1080, 1151, 1152, 1153, 1344,
          1728, 1919, 1920, 1921, 2047, 2048]


@pytest.mark.parametrize("passes", [1, 2, 3, 7])
@pytest.mark.parametrize("strength,gain", [(0.0, 0.0), (0.4, 1.0), (12.0, 0.0), (61.0, 0.5), (100.0, 1.0)])
def test_line_lengths(ctx, orc, strength, gain, passes):
    for W in WIDTHS:
        _check(ctx, orc, "h", W, 5, strength, gain, passes)


@pytest.mark.parametrize("passes", [1, 3, 4])
@pytest.mark.parametrize("W,H", [(1920, 1027), (600, 2047), (321, 2048), (64, 1030)])
def test_many_lines(ctx, orc, W, H, passes):
    _check(ctx, orc, "h", W, H, 12.0, 0.0, passes)


@pytest.mark.parametrize("passes", [1, 2, 3, 64])
@pytest.mark.parametrize("kind,W,H", [("v", 1920, 1080), ("v", 1028, 516), ("2d", 2048, 320), ("2d", 4, 8)])
def test_transposed_stores(ctx, orc, kind, W, H, passes):
    _check(ctx, orc, kind, W, H, 3.0, 0.25, passes)


@pytest.mark.parametrize("value", [0, 0xffffffff])
def test_flat_images(ctx, orc, value):
    """sums at their least and their greatest"""
    W, H = 1925, 6
    for strength, gain in [(0.0, 1.0), (0.2, 1.0), (100.0, 1.0), (100.0, 0.0)]:
        n = W * H
        src = np.full(n + 4, value, np.uint32)
        src[n:] = 0
        want, s0, s1 = (np.zeros(n + 4, np.uint32) for _ in range(3))
        orc.orc_blur26_h(P(want), P(src), W, H, strength, gain, 3, P(s0), P(s1))
        d, s = ctx.empty(n), ctx.upload(src[:n])
        ctx.blur26_h(d, s, W, H, strength, gain, 3)
        assert np.array_equal(d.numpy(), want[:n]), (strength, gain)
        ctx.free(s)
        ctx.free(d)


def _span_strength(W, span, alpha):
    """the strength whose radius on a line of W pixels is span + alpha"""
    return 100.0 * (span + alpha) / ((W - 2) // 2)


def _both_orders(ctx, orc, src, W, H, strength, gain, passes, before=lambda: None):
    n = W * H
    for kind in ("h", "v"):
        w, h = (W, H) if kind == "h" else (H, W)
        img = np.zeros(n + 4, np.uint32)
        img[:n] = (src if kind == "h" else src.T).reshape(-1)
        want, s0, s1 = (np.zeros(n + 4, np.uint32) for _ in range(3))
        {"h": orc.orc_blur26_h, "v": orc.orc_blur26_v}[kind](
            P(want), P(img), w, h, strength, gain, passes, P(s0), P(s1))
        d, s = ctx.empty(n), ctx.upload(img[:n])
        before()
        {"h": ctx.blur26_h, "v": ctx.blur26_v}[kind](d, s, w, h, strength, gain, passes)
        got = d.numpy()
        ctx.free(s)
        ctx.free(d)
        bad = np.nonzero(got != want[:n])[0]
        assert len(bad) == 0, (kind, len(bad), int(bad[0]) // w, int(bad[0]) % w)


@pytest.mark.parametrize("gain", [0.0, 1.0])
@pytest.mark.parametrize("span", [1, 3, 15, 63, 127, 255, 256, 257, 500])
def test_sums_above_the_flat_image(ctx, orc, span, gain):
    """the terms subtracted are rounded down, so a line that is random where
    they come from and 255 elsewhere has sums above the flat image's: at a span
    of 256 they pass 2^17"""
    W, H = 1024, 8
    rng = np.random.default_rng(span)
    line = np.full((H, W, 4), 255, np.uint8)
    line[:, 1:span] = rng.integers(0, 256, (H, span - 1, 4))
    line[:, span:span + 2] = 0
    src = np.ascontiguousarray(line).view(np.uint32).reshape(H, W)
    strength = _span_strength(W, span, 0.997) if span < 500 else 100.0
    for passes in (1, 2):
        print("sums", span, gain, passes, flush=True)
        _both_orders(ctx, orc, src, W, H, strength, gain, passes)


# two or three passes of a launch whose halo waves hold barely the pixels
# needed, for 3, 5, 7 and 9 pixels a lane
@pytest.mark.parametrize("W,H,span,passes", [
    (1024, 40, 189, 2), (1024, 40, 190, 2), (1024, 40, 382, 2), (1024, 300, 190, 2), (1024, 40, 191, 2),
    (1920, 1032, 315, 2), (1920, 1032, 317, 2), (1920, 1032, 318, 2), (1344, 1032, 443, 2), (1344, 1032, 446, 2),
    (1024, 40, 94, 3), (1920, 1032, 158, 3), (1600, 1032, 284, 3), (1600, 1032, 286, 3)])
def test_halo_of_the_next_line(ctx, orc, W, H, span, passes):
    """every launch after one of another kernel that leaves pixels in LDS"""
    rng = np.random.default_rng(W + span)
    noise = rng.integers(0, 1 << 32, (H, W), dtype=np.uint64).astype(np.uint32)
    dark = noise & np.uint32(0x1f1f1f1f)
    lines = rng.integers(0, 1 << 32, (2048, 2000), dtype=np.uint64).astype(np.uint32).reshape(-1)
    t = ctx.upload(lines)

    def leave_pixels():
        ctx.blur07_inplace_batch([t], [7.5 / 255.0], 2000, 2048, 1)

    print("halo", W, H, span, passes, flush=True)
    for src in (noise, dark):
        _both_orders(ctx, orc, src, W, H, _span_strength(W, span, 0.4), 0.0, passes, leave_pixels)
    ctx.free(t)
