"""The layout of a library's tables in their one allocation, on the CPU.

Each table begins on 256 bytes: K nearest reads the block layout 64 values at a
time, which are two cache lines of 128 bytes from such a start and three from
any other.  No two tables overlap, and all lie inside the allocation.
"""
import ctypes

import pytest

NAMES = ["lab4", "box", "L", "A", "B", "pL", "pA", "pB", "pidx", "bytes"]


class Layout(ctypes.Structure):
    _fields_ = [(k, ctypes.c_size_t) for k in NAMES]


@pytest.mark.parametrize("n", [0, 1, 2, 63, 64, 65, 1000, 1500, 2500, 5000, 10000, 33847, 1 << 20])
def test_aligned_and_apart(mh, n):
    fn = ctypes.CDLL(mh.LIB_PATH)._ZN2mh4host12table_layoutEi
    fn.restype = Layout
    t = fn(ctypes.c_int32(n))
    m = max(n, 1)
    blocks = (m + 63) // 64
    size = {"lab4": 16 * m, "box": 32 * blocks, "L": 4 * m, "A": 4 * m, "B": 4 * m}
    size.update({k: 256 * blocks for k in ("pL", "pA", "pB", "pidx")})
    end = 0
    for k in NAMES[:-1]:
        at = getattr(t, k)
        assert at % 256 == 0 and at >= end
        end = at + size[k]
    assert end <= t.bytes < end + 256
