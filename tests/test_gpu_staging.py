"""Large host copies through the pinned buffers (mh_stage.hip), against the oracle.

Images of several sizes whose spans begin and end inside, at and across the
buffers' chunks: one image of several chunks, many small ones in each, totals
just under and over the least that is staged and a whole number of chunks, a
span of the smallest size, a read-only and a non-contiguous array.  The Lab
means of all images must be those of each alone, bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    [(1, 1)] * 3,
    [(512, 682), (1, 2)],                      # 1 MiB - 1,024 and 6 bytes more
    [(1024, 1024)] * 2 + [(37, 41)] * 5,       # 6 MiB and a little
    [(512, 2048)] * 8,                         # 24 MiB: six whole chunks
    [(700, 501)] * 9 + [(3, 5)] + [(1200, 1100)],
    [(37, 41)] * 900 + [(64, 64)] * 300,
]


@pytest.mark.parametrize("sizes", CASES)
def test_images_from_where_they_lie(ctx, orc, sizes):
    rng = np.random.default_rng(len(sizes))
    images = [rng.integers(0, 256, (h, w, 3), dtype=np.uint8) for h, w in sizes]
    images[0].setflags(write=False)
    images[-1] = np.asfortranarray(images[-1])
    want = np.stack([orc.stack_lab_means(np.ascontiguousarray(im)[None])[0] for im in images])
    got = ctx.average_lab_many(images)
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    lib = ctx.library_from_images(images)
    np.testing.assert_array_equal(lib.lab().view(np.uint32), want.view(np.uint32))
    lib.close()
