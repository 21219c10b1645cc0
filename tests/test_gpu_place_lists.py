"""The placement chain over prepared candidate lists (k_place.hip), against the oracle.

The lists are used where no per-cell output is asked for, so the cases call
mh_place without them.  They stand at the edges of the chain's forms: grids
around 48 columns (who bans the up neighbour) and of a few, cell counts that
are no multiple of a group, libraries around 64 materials (whose lists keep
exhausted candidates), of one tile, with duplicate Labs, with the Labs out of
LDS and with no place for lists at all; limits that reset every cell, often and
never, around the 16 bits of a packed count, and counts that a caller has set.
Every result is a whole number and equal to the oracle's.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # gw, gh, n, limit, weight, distinct Labs, counts given
    (3, 41, 80, 2, 0.5, 80, False),
    (4, 30, 700, 3, 40.0, 40, False),
    (13, 11, 65, 1, 0.25, 65, False),
    (47, 9, 120, 3, 5.0, 120, False),
    (48, 9, 120, 3, 5.0, 120, False),
    (49, 9, 64, 6, 0.25, 64, False),
    (49, 9, 64, 2, 0.25, 20, False),
    (60, 7, 1, 3, 0.3, 1, False),
    (60, 7, 2, 0, 0.3, 2, False),
    (61, 11, 300, 0, 0.3, 300, False),
    (131, 5, 101, 1, 0.5, 101, False),
    (97, 13, 500, 65535, 0.3, 500, False),
    (97, 13, 500, 65536, 0.3, 500, False),
    (50, 28, 200, 70000, 0.3, 200, True),
    (20, 28, 64, 3, 0.3, 64, True),
    (97, 13, 500, 3, 0.0, 500, False),
    (97, 13, 500, 3, 1e6, 30, False),
    (64, 30, 9000, 3, 0.5, 3000, False),
    (64, 12, 34000, 1, 0.5, 34000, False),
    (300, 40, 900, 2, 0.3, 900, False),
]


@pytest.mark.parametrize("score_mode", [0, 1])
@pytest.mark.parametrize("gw,gh,n,limit,weight,distinct,given", CASES)
def test_lists(mh, ctx, orc, gw, gh, n, limit, weight, distinct, given, score_mode):
    rng = np.random.default_rng(gw * 1009 + n)
    lab = (rng.random((n, 3)) * [100, 60, 60] - [0, 30, 30]).astype(np.float32)
    lab = lab[np.arange(n) % distinct]
    # a smooth target: neighbouring cells want the same materials
    y, x = np.mgrid[0:gh, 0:gw]
    cl = np.stack([100 * x / gw, 60 * y / gh - 30, 30 * (x + y) / (gw + gh) - 15], -1)
    cl = (cl + rng.normal(0, 1.5, cl.shape)).astype(np.float32).reshape(-1, 3)
    usage = rng.integers(max(limit - 3, 0), limit + 2, n) if given else np.zeros(n)
    usage = usage.astype(np.uint32)
    want = orc.place(lab, cl, gw, gh, limit, weight, usage=usage, score_mode=score_mode)
    lib = ctx.library_from_lab(lab)
    grid, got_usage = np.full(gw * gh, -1, np.int32), usage.copy()
    stats, params = mh.PlaceStats(), mh.PlaceParams(gw, gh, limit, weight, score_mode)
    mh._check(ctx.lib.mh_place(ctx.h, lib.h, mh._ptr(cl), ctypes.byref(params), None, 0, mh._ptr(grid),
                               mh._ptr(got_usage), None, None, None, ctypes.byref(stats)))
    lib.close()
    np.testing.assert_array_equal(grid, want["grid"])
    np.testing.assert_array_equal(got_usage, want["usage"])
    assert stats.as_dict() == want["stats"]
