"""The bounded division's quotients equal n / d bit for bit (quotients.hip): 2^30
random pairs and three times 2^30 around the halfway cases of 2^30 divisors just
below a power of two and of as many random ones."""
import ctypes
import os

import pytest

pytestmark = pytest.mark.gpu
LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "le2d_amd", "lib",
                   "libquotients.so")


@pytest.mark.parametrize("kind", [0, 1, 2])
def test_quotients(kind):
    lib = ctypes.CDLL(LIB)
    lib.check_quotients.argtypes = [ctypes.c_int, ctypes.c_long, ctypes.c_ulonglong,
                                    ctypes.POINTER(ctypes.c_ulonglong)]
    out = (ctypes.c_ulonglong * 3)()
    assert lib.check_quotients(kind, 1 << 30, 12345, out) == 0
    assert out[0] == 0, [hex(v) for v in out]
