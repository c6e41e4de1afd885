"""st_sqrt, the square root of the raymarched effects' steps, against the
correctly rounded root: every float of the range in which it does not call
sqrtf, on the device, and both exponent parities against numpy's."""
import ctypes as C

import numpy as np
import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sweep(ctx):
    lib = C.CDLL(str(ROOT / "tests" / "native" / "sqrt_sweep.so"))
    lib.sqrt_sweep.restype = C.c_longlong
    lib.sqrt_sweep.argtypes = [C.c_uint32, C.c_uint32, C.c_void_p]
    return lib.sqrt_sweep


def test_every_float_of_the_range(sweep):
    # 2^-96 .. 2^96, and an exponent either side
    for first in range(127 - 97, 127 + 97, 32):
        assert sweep(first, min(first + 31, 127 + 97), None) == 0, first


def test_other_floats(sweep):
    assert sweep(0, 3, None) == 0      # 0 and subnormal numbers
    assert sweep(250, 254, None) == 0


@pytest.mark.parametrize("exponent", [127, 128])
def test_against_the_host(sweep, exponent):
    out = np.zeros(1 << 23, np.uint32)
    assert sweep(exponent, exponent, out.ctypes.data) == 0
    x = (np.arange(1 << 23, dtype=np.uint32) | np.uint32(exponent << 23)).view(np.float32)
    assert np.array_equal(out, np.sqrt(x).view(np.uint32))
