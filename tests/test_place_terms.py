"""Which libraries have their largest adjacency terms, and which runs read them.

The placement's prepared lists (k_place.hip) take a candidate as safe from a
bound on its penalty, the material's largest adjacency term to another
material.  A library computes those terms when it is made, if any grid can take
it in lists; the LDS that lists need is least at 48 columns, not at one.  A run
on lists without the terms would leave the penalties out without a sign of it.

The rule is checked on the CPU over all widths and the sizes where lists stop
fitting 160 KiB; the GPU cases stand at those sizes and are equal to the oracle.
"""
import ctypes

import numpy as np
import pytest

LDS = 160 * 1024
PLAIN, LISTS = 0, 1


def _rules(mh):
    lib = ctypes.CDLL(mh.LIB_PATH)
    form = lib._ZN2mh11raster_formEiibbm   # (grid_w, n, labs, terms, max_lds)
    form.argtypes = [ctypes.c_int32, ctypes.c_int32] + [ctypes.c_bool] * 2 + [ctypes.c_size_t]
    takes = lib._ZN2mh11lists_takenEim     # (n, max_lds)
    takes.restype = ctypes.c_bool
    takes.argtypes = [ctypes.c_int32, ctypes.c_size_t]
    words = lib._ZN2mh22place_raster_lds_bytesEiii
    words.restype = ctypes.c_size_t
    return form, takes, words


def test_lists_only_with_terms(mh):
    form, takes, words = _rules(mh)
    for n in [1, 64, 65, 1500, 9000, 33000] + list(range(33700, 34000, 3)) + [33827, 33828, 33847, 33848, 36000]:
        has = takes(n, LDS)
        for gw in list(range(1, 140)) + [200, 500, 1000, 4000]:
            for labs in (False, True):
                # whatever the library has, a run without terms is not on lists
                assert form(gw, n, labs, False, LDS) < LISTS
                # and where lists fit, the library has the terms
                fits = gw >= 3 and words(gw, n, LISTS) <= LDS
                assert (form(gw, n, labs, has, LDS) >= LISTS) == fits, (gw, n)


CASES = [
    # gw, gh, n, limit, weight
    (48, 27, 33840, 3, 0.5),
    (48, 27, 33840, 3, 5.0),
    (67, 9, 33828, 3, 0.5),
    (67, 9, 33828, 3, 5.0),
    (48, 9, 33847, 2, 0.5),
    (48, 9, 33847, 2, 5.0),
    (48, 9, 33848, 2, 5.0),
    (68, 9, 33828, 2, 5.0),
    (20, 9, 33827, 2, 5.0),
]


@pytest.mark.gpu
@pytest.mark.parametrize("score_mode", [0, 1])
@pytest.mark.parametrize("gw,gh,n,limit,weight", CASES)
def test_sizes_where_lists_stop_fitting(mh, ctx, orc, gw, gh, n, limit, weight, score_mode):
    rng = np.random.default_rng(gw * 1009 + n)
    lab = (rng.random((n, 3)) * [100, 60, 60] - [0, 30, 30]).astype(np.float32)
    y, x = np.mgrid[0:gh, 0:gw]
    cl = np.stack([100 * x / gw, 60 * y / gh - 30, 30 * (x + y) / (gw + gh) - 15], -1)
    cl = (cl + rng.normal(0, 1.5, cl.shape)).astype(np.float32).reshape(-1, 3)
    want = orc.place(lab, cl, gw, gh, limit, weight, score_mode=score_mode)
    free = orc.place(lab, cl, gw, gh, limit, 0.0, score_mode=score_mode)
    assert np.any(want["grid"] != free["grid"])  # penalties decide some cells
    lib = ctx.library_from_lab(lab)
    grid, usage = np.full(gw * gh, -1, np.int32), np.zeros(n, np.uint32)
    stats, params = mh.PlaceStats(), mh.PlaceParams(gw, gh, limit, weight, score_mode)
    mh._check(ctx.lib.mh_place(ctx.h, lib.h, mh._ptr(cl), ctypes.byref(params), None, 0, mh._ptr(grid),
                               mh._ptr(usage), None, None, None, ctypes.byref(stats)))
    lib.close()
    np.testing.assert_array_equal(grid, want["grid"])
    np.testing.assert_array_equal(usage, want["usage"])
    assert stats.as_dict() == want["stats"]
