"""The placement chain that reads whole rows (k_place.hip: raster_plain), against the oracle.

Libraries whose counts leave LDS no place for lists (33,848 to 40,700
materials) and grids of one or two columns.  A cell's first candidate wins at
once when the others lie beyond its largest possible score, so the weights run
from one that no distance is within to one that every distance is within, with
exact ties: duplicate Labs at weight 0 and above.  Whole numbers, equal.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # gw, gh, n, distinct Labs, limit
    (40, 11, 33848, 33848, 3),
    (40, 11, 33848, 900, 1),
    (5, 9, 40700, 40700, 2),
    (1, 97, 300, 60, 2),
    (2, 51, 150, 150, 1),
    (2, 51, 3, 3, 1),
    (1, 97, 130, 130, 0),
]


@pytest.mark.parametrize("score_mode", [0, 1])
@pytest.mark.parametrize("weight", [-1.0, 0.0, 1e-6, 0.25, 30.0, 1e6, 3e38])
@pytest.mark.parametrize("gw,gh,n,distinct,limit", CASES)
def test_plain(mh, ctx, orc, gw, gh, n, distinct, limit, weight, score_mode):
    rng = np.random.default_rng(gw * 1009 + n)
    lab = (rng.random((n, 3)) * [100, 60, 60] - [0, 30, 30]).astype(np.float32)[np.arange(n) % distinct]
    y, x = np.mgrid[0:gh, 0:gw]
    cl = np.stack([100 * x / gw, 60 * y / gh - 30, 30 * (x + y) / (gw + gh) - 15], -1)
    cl = (cl + rng.normal(0, 1.5, cl.shape)).astype(np.float32).reshape(-1, 3)
    want = orc.place(lab, cl, gw, gh, limit, weight, score_mode=score_mode)
    lib = ctx.library_from_lab(lab)
    got = ctx.place(lib, cl, gw, gh, limit, weight, score_mode=score_mode)
    lib.close()
    for k in ("grid", "usage", "stage", "dist", "score"):
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)
    assert got["stats"] == want["stats"]
