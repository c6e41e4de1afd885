"""The FX maps' cosine look-up (an entry and its step in one read, the index of
an angle at or above 2^31 being 0) and their square root: Plasma, whose whole
arithmetic is the reference's, from ordinary times to such that every angle is
past the index's range, bit for bit against the oracle; and at sizes whose maps
no tile divides."""
import numpy as np
import pytest

import oracles
from cookiedough_amd import _lib
from cookiedough_amd import workloads as wl
from test_gpu_shadertoy import gpu_map, orc_map
from oracles import P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(320, 180), (88, 66)])
@pytest.mark.parametrize("time", [0.0, 17.5, -17.5, 1e4, 3e6, 1.1e8, 1e12, 1e30])
def test_plasma_at_any_time(ctx, orc, time, W, H):
    lut = np.zeros(2049, np.float32)
    orc.orc_cos_lut(P(lut))
    tex = np.zeros(1 << 20, np.uint32)
    prm = _lib.ST_PARAMS["plasma"](time=time, **wl.ST_DEMO["plasma"])
    got, _ = gpu_map(ctx, "plasma", prm, W, H, False)
    want, _ = orc_map(orc, (lut, tex, tex, None), oracles.ST_IDS["plasma"], prm, W, H)
    assert np.array_equal(got, want), (time, int((got != want).sum()))
