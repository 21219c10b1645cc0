"""Cells one, two and three pixels wide in the composite (k_composite.hip), against the oracle.

Rows around the number of cells that a block of one job's launch (256 threads)
and of the batched launch (64, 128, 256) covers at these widths; with and
without the colour adjustment.  The job alone and in a batch of every block
size.  Bytes equal the oracle's.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("strength", [0.0, 0.4])
@pytest.mark.parametrize("gw,gh,tw,th", [(1023, 2, 1, 1), (1025, 1, 1, 2), (513, 2, 1, 3), (511, 2, 2, 1), (513, 1, 2, 3),
                                         (257, 2, 3, 2), (5, 3, 1, 64), (3, 3, 2, 5)])
def test_narrow_cells(mh, ctx, orc, gw, gh, tw, th, strength):
    rng = np.random.default_rng(gw * 131 + tw)
    mats = rng.integers(0, 256, (60, th + 3, tw + 2, 3)).astype(np.uint8)
    target = rng.integers(0, 256, (gh * th, gw * tw, 3)).astype(np.uint8)
    lib = ctx.library_from_pixels(mats)
    p = mh.JobParams(gw, gh, 100000, 0.25, strength, 0, 0, 100.0, 0.99995, 0, 0)
    d_t = ctx.to_device(target)
    batch = ctx.batch([ctx.job(lib, d_t, gw * tw, gh * th, p)] * 3)
    one = ctx.generate(lib, target, gw, gh, 100000, 0.25, strength, enable_optimization=False)
    want = orc.composite(target, mats, one["grid"], gw, gh, strength)
    np.testing.assert_array_equal(one["image"], want)
    for threads in (64, 128, 256):
        batch.set_tuning(composite_threads=(threads, threads))
        batch.run()
        ctx.synchronize()
        for i in range(3):
            np.testing.assert_array_equal(ctx.to_host(batch.outputs(i)[1], want.shape, np.uint8), want)
    batch.close()
    ctx.device_free(d_t)
    lib.close()
