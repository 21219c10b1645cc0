"""Per-cell outputs of mh_place in raster order, against the oracle.

They are made from the grid that the chain leaves and from the stages of its
resets (k_place.hip: place_outputs_kernel), whichever outputs are asked for.
The cases: lists with the Labs in LDS and out of it, one and two columns, a
library with no place for lists; no penalty; limits that reset every cell (with
candidates left, and with one tile none), often and never; counts that a caller
has set; cell counts that are no multiple of a block's four.  Whole numbers are
equal, distances and scores bit for bit (the oracle's f32 operations).
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # gw, gh, n, limit, weight, counts given
    (20, 15, 1000, 3, 0.25, False),
    (49, 9, 64, 2, 0.25, False),
    (50, 11, 120, 0, 0.5, False),
    (50, 11, 1, 3, 0.5, False),
    (61, 7, 2, 1, 0.0, False),
    (61, 7, 90, 3, 5.0, True),
    (64, 30, 9000, 3, 0.5, False),
    (41, 5, 34000, 1, 0.5, False),
    (1, 203, 70, 2, 0.5, False),
    (2, 101, 70, 2, 0.5, False),
    (7, 3, 41500, 2, 0.5, False),
    (5, 1, 3, 1, 0.25, False),
]
WANTED = [("stage",), ("stage", "dist"), ("score",), ("dist",), ("stage", "dist", "score")]


@pytest.mark.parametrize("score_mode", [0, 1])
@pytest.mark.parametrize("gw,gh,n,limit,weight,given", CASES)
def test_outputs(mh, ctx, orc, gw, gh, n, limit, weight, given, score_mode):
    rng = np.random.default_rng(gw * 1009 + n)
    lab = (rng.random((n, 3)) * [100, 60, 60] - [0, 30, 30]).astype(np.float32)
    y, x = np.mgrid[0:gh, 0:gw]
    cl = np.stack([100 * x / gw, 60 * y / gh - 30, 30 * (x + y) / (gw + gh) - 15], -1)
    cl = (cl + rng.normal(0, 1.5, cl.shape)).astype(np.float32).reshape(-1, 3)
    usage = (rng.integers(max(limit - 2, 0), limit + 2, n) if given else np.zeros(n)).astype(np.uint32)
    want = orc.place(lab, cl, gw, gh, limit, weight, usage=usage, score_mode=score_mode)
    lib = ctx.library_from_lab(lab)
    params = mh.PlaceParams(gw, gh, limit, weight, score_mode)
    for names in WANTED:
        grid, got_usage, stats = np.full(gw * gh, -1, np.int32), usage.copy(), mh.PlaceStats()
        out = {"stage": np.full(gw * gh, 255, np.uint8), "dist": np.full(gw * gh, np.nan, np.float32),
               "score": np.full(gw * gh, np.nan, np.float32)}
        ptrs = [mh._ptr(out[k]) if k in names else None for k in ("stage", "dist", "score")]
        mh._check(ctx.lib.mh_place(ctx.h, lib.h, mh._ptr(cl), ctypes.byref(params), None, 0,
                                   mh._ptr(grid), mh._ptr(got_usage), *ptrs, ctypes.byref(stats)))
        np.testing.assert_array_equal(grid, want["grid"])
        np.testing.assert_array_equal(got_usage, want["usage"])
        assert stats.as_dict() == want["stats"]
        for k in names:
            np.testing.assert_array_equal(out[k].view(np.uint8), want[k].view(np.uint8), err_msg=f"{names} {k}")
    lib.close()


def test_no_materials(mh, ctx):
    lib = ctx.library_from_lab(np.zeros((0, 3), np.float32))
    got = ctx.place(lib, np.zeros((12, 3), np.float32), 4, 3, 2, 0.5)
    assert (got["grid"] == -1).all() and (got["stage"] == 255).all()
    assert np.isnan(got["dist"]).all() and np.isnan(got["score"]).all()
    lib.close()
