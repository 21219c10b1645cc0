"""Cells one pixel wide (k_lab.hip divides a pixel's index by the width), against the oracle.

Their Lab means, and whole jobs of them with the colour adjustment (whose target
averages come from the same kernel), alone, in a batch and as materials of one
column.  Values equal bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gw,gh,tw,th", [(5, 3, 1, 64), (33, 2, 1, 2), (7, 4, 1, 1), (300, 3, 1, 300), (9, 2, 2, 33), (1, 1, 1, 9),
                                         (300, 220, 1, 2)])
def test_narrow_cells(mh, ctx, orc, gw, gh, tw, th):
    rng = np.random.default_rng(gw * 131 + th)
    target = rng.integers(0, 256, (gh * th, gw * tw, 3)).astype(np.uint8)
    cells = target.reshape(gh, th, gw, tw, 3).transpose(0, 2, 1, 3, 4).reshape(gw * gh, th, tw, 3)
    want_lab = orc.stack_lab_means(np.ascontiguousarray(cells))
    np.testing.assert_array_equal(ctx.cell_lab_means(target, gw, gh).view(np.uint32), want_lab.view(np.uint32))
    if gw * gh > 2000:
        return
    mats = rng.integers(0, 256, (40, th + 3, 1, 3)).astype(np.uint8)
    lib = ctx.library_from_pixels(mats)
    np.testing.assert_array_equal(lib.lab().view(np.uint32), orc.stack_lab_means(mats).view(np.uint32))
    want = orc.generate(target, mats, gw, gh, 100000, 0.25, 0.4, True, 50, seed=3)
    got = ctx.generate(lib, target, gw, gh, 100000, 0.25, 0.4, True, 50, seed=3)
    np.testing.assert_array_equal(got["grid"], want["grid"])
    np.testing.assert_array_equal(got["image"], want["image"])
    d_t = ctx.to_device(target)
    batch = ctx.batch([ctx.job(lib, d_t, gw * tw, gh * th,
                               mh.JobParams(gw, gh, 100000, 0.25, 0.4, 1, 50, 100.0, 0.99995, 3, 0))] * 2)
    batch.run()
    ctx.synchronize()
    for i in range(2):
        np.testing.assert_array_equal(ctx.to_host(batch.outputs(i)[1], want["image"].shape, np.uint8), want["image"])
    batch.close()
    ctx.device_free(d_t)
    lib.close()
