"""The in-place 2007 blur as a scan (code/deprecated/boxblur.cpp with pDest ==
pSrc): a step is a clamped addition, clamped additions compose, so a chunk of
steps is a prefix scan.  Bit-exact against the oracle at every chunk length
(medians 4, 6, 8, 10, 12, 16 and just above), even and odd spans, lines no
longer than the span and up to the longest LDS holds, line counts that do not
fill a block, images that drive the accumulator into both clamps, and both
sides of the batch size where the other kernels take over."""
import numpy as np
import pytest

from helpers import rand_img
from oracles import P


def strength_of_span(span):
    return (span + 0.5) / 255.0


def _image(kind, n, seed):
    rng = np.random.default_rng(seed)
    if kind == "noise":
        return rand_img(seed, n)
    # long runs of 0 and 255 per channel
    run = int(rng.integers(3, 300))
    v = np.repeat(rng.integers(0, 2, (n // run + 1, 4)).astype(np.uint8) * 255, run, axis=0)[:n]
    return np.ascontiguousarray(v).view(np.uint32).reshape(-1)


def _check(ctx, orc, W, H, n, spans, passes, kind, seed):
    f = {1: orc.orc_blur07_h, 2: orc.orc_blur07_v}[passes]
    srcs = [_image(kind, W * H, seed + j) for j in range(n)]
    dev = [ctx.upload(s) for s in srcs]
    st = [strength_of_span(spans[j % len(spans)]) for j in range(n)]
    ctx.blur07_inplace_batch(dev, st, W, H, passes)
    ctx.sync()
    for j in range(n):
        want = srcs[j].copy()
        f(P(want), P(want), W, H, st[j], 8)
        assert np.array_equal(dev[j].numpy(), want), (W, H, j, st[j], passes, kind)
    for d in dev:
        ctx.free(d)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["noise", "runs"])
@pytest.mark.parametrize("passes", [1, 2])
@pytest.mark.parametrize("span", [7, 8, 9, 11, 12, 15, 16, 19, 20, 21, 23, 24, 31, 32, 33, 82, 254, 255])
def test_every_chunk_length(ctx, orc, span, passes, kind):
    # the line as long as the span, a little longer, many chunks
    for k, length in enumerate((span, span + 1, span + 17, 2 * span + 130, 777)):
        W, H = (length, 5) if passes == 1 else (5, length)
        _check(ctx, orc, W, H, 1, [span], passes, kind, 1000 * span + k)


@pytest.mark.gpu
@pytest.mark.parametrize("passes", [1, 2])
@pytest.mark.parametrize("length,lines", [(4079, 6), (4080, 6), (8175, 3), (8176, 3), (16367, 2), (16368, 2)])
def test_longest_lines(ctx, orc, length, lines, passes):
    W, H = (length, lines) if passes == 1 else (lines, length)
    _check(ctx, orc, W, H, 1, [76], passes, "noise", 7)


# 256 CUs: 2560 lines at 4 steps a chunk; 17920 lines of 96 pixels are past the
# limit at 16 (test_limits_by_length)
@pytest.mark.gpu
@pytest.mark.parametrize("span,lines,n", [(8, 1280, 2), (8, 1281, 2), (40, 1280, 14), (40, 1281, 14)])
def test_batch_limit(ctx, orc, span, lines, n):
    _check(ctx, orc, 96, lines, n, [span, span + 3], 1, "runs", 90)


# 256 CUs again, where the scan gives way sooner: rows of 96 pixels at 16 steps
# from 7168 lines on, columns of 96 at 10 steps from 7447, columns of 16000
# pixels, two blocks of one a CU, from 716 at 4 steps
@pytest.mark.gpu
@pytest.mark.parametrize("W,H,n,span,passes", [
    (96, 1024, 7, 40, 1), (96, 1025, 7, 40, 1), (1063, 96, 7, 22, 2), (1064, 96, 7, 22, 2),
    (716, 16000, 1, 10, 2), (717, 16000, 1, 10, 2)])
def test_limits_by_length(ctx, orc, W, H, n, span, passes):
    _check(ctx, orc, W, H, n, [span, span + 3], passes, "noise", 91)


def test_clamped_additions_compose():
    """the scan's composition against the reference's two saturating steps"""
    rng = np.random.default_rng(5)
    n, steps = 4000, 16
    a = rng.integers(0, 256, (steps, n)) * rng.integers(0, 2, (steps, n))
    s = rng.integers(0, 256, (steps, n)) * rng.integers(0, 2, (steps, n))
    acc = np.concatenate([rng.integers(0, 600, n // 2), 65535 - rng.integers(0, 600, n // 2)])
    d, lo, hi = np.zeros(n, int), np.full(n, -(1 << 28)), np.full(n, 1 << 28)
    want = acc.copy()
    for k in range(steps):
        want = np.maximum(np.minimum(want + a[k], 65535) - s[k], 0)
        d2, h2 = a[k] - s[k], 65535 - s[k]
        d, lo, hi = d + d2, np.clip(lo + d2, 0, h2), np.clip(hi + d2, 0, h2)
        assert np.array_equal(np.clip(acc + d, lo, hi), want)
