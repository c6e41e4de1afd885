"""The 2026 blur's sums as factors of a 24-bit multiply (cookiedough_amd/csrc/
k_blur26.hip, horz): no line's sum passes (2 span + 2) * 255 + span + 1, and that
bound's shift and the scale's leave both factors inside 24 bits with the sign,
for every span."""
import numpy as np
import pytest


def bound(span):
    return (2 * span + 2) * 255 + span + 1


def test_factors_fit_24_bits():
    for span in range(501):
        sum_shift = min(10, 23 - bound(span).bit_length())
        scale_shift = 10 - sum_shift
        assert sum_shift >= 0
        assert bound(span) << sum_shift < 1 << 23
        assert (1 << 22) // (span + 1) << scale_shift < 1 << 23


@pytest.mark.parametrize("span", [0, 1, 2, 15, 63, 127, 255, 256, 257, 500])
def test_sums_stay_below_the_bound(span):
    """HorzBlur32's running sum (code/boxblur.cpp:126-211) over lines whose
    subtracted terms round down as often as they can"""
    rng = np.random.default_rng(span)
    L, most = 4 * span + 20, 0
    for alpha in (0, 1, 255, 32768, 65279, 65300, 65400, 65535):
        for low in (rng.integers(0, 256, span + 2), np.arange(span + 2) % 2 * 255, np.arange(span + 2) % 256):
            p = np.full(L + 2, 255, np.int64)
            p[1:span + 1] = low[1:span + 1]
            p[max(span, 1):span + 2] = 0
            T = (p[:-1] + ((p[1:] - p[:-1]) * alpha >> 16))[:L + 1]
            C = np.concatenate([[0], np.cumsum(T)])
            o = np.arange(L)
            s0 = p[:span].sum() + (p[span] * alpha >> 16)
            S = s0 + C[np.minimum(span + o, L) + 1] - C[span + 1] - C[np.maximum(o - span, 0)]
            most = max(most, int(S.max()))
    assert most <= bound(span)
    if span == 256:
        assert most >= 1 << 17  # the case that (2 span + 2) * 255 alone misses
