"""The binding's table of host images (mosaic_hip._image_table), on the CPU.

Small images (under 8 KiB on average) are copied into one array, others are
named where they lie.  Either way base + offset holds each image's bytes.
"""
import ctypes

import numpy as np
import pytest

CASES = [
    [],
    [(1, 1)],
    [(3, 5), (1, 2), (40, 17)],
    [(52, 52)] * 3 + [(53, 52)],       # 8,112 bytes and one of 8,268: copied
    [(53, 52)] * 3,                    # in place
    [(1, 1)] * 9 + [(200, 137)],       # small but for one: on average 8,222, in place
    [(1, 1)] * 10 + [(200, 137)],      # 7,475, copied
]


@pytest.mark.parametrize("sizes", CASES)
def test_bytes(mh, sizes):
    rng = np.random.default_rng(len(sizes))
    images = [rng.integers(0, 256, (h, w, 3), dtype=np.uint8) for h, w in sizes]
    if len(images) > 1:
        images[0].setflags(write=False)
        images[-1] = np.asfortranarray(images[-1])
    keep, base, off, w, h = mh._image_table(images)
    assert off.dtype == np.int64 and w.dtype == np.int32 and h.dtype == np.int32
    assert len(off) == len(w) == len(h) == len(images)
    assert (off >= 0).all()
    for i, im in enumerate(images):
        assert (h[i], w[i]) == im.shape[:2]
        p = ctypes.addressof((ctypes.c_uint8 * im.size).from_address(base.value + int(off[i])))
        assert ctypes.string_at(p, im.size) == np.ascontiguousarray(im).tobytes()
    copied = bool(images) and sum(im.size for im in images) < 8192 * len(images)
    assert isinstance(keep, np.ndarray) == copied
