"""Short forms of IEEE operations in the device code (mh_device.hpp), on the device.

The hardware's estimates corrected by fused residual steps stand for a square
root, reciprocals and quotients, and costs, annealing and placement rely on
their bits.  Every non-negative float is compared for an adjacency term, every
divisor of the colour adjustment's range for its reciprocal and eight quotients
(device_test/identities.hip).  None may differ.
"""
import ctypes
import os

import pytest

pytestmark = pytest.mark.gpu


def test_no_bit_differs(mh):
    lib = ctypes.CDLL(os.path.join(os.path.dirname(mh.LIB_PATH), "libmosaic_hip_test.so"))
    bad = (ctypes.c_uint32 * 3)()
    assert lib.mh_test_identities(ctypes.c_uint32(4), bad) == 0
    assert list(bad) == [0, 0, 0], "terms, reciprocals, quotients that differ"
