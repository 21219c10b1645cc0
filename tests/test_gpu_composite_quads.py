"""The composite's quads (k_composite.hip), against the oracle.

Cell widths of one to nine pixels and around 16 (one quad to a cell, short last
quads of every length, none), rows that end inside a block and that fill
several, empty cells, materials of extreme colours (greys, black, white, pure
hues: the divisions' and the sextants' edges), and strengths of the colour
adjustment down to values whose hue shifts are below the division's short
cut.  Bytes equal the oracle's.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EXTREMES = [[0, 0, 0], [255, 255, 255], [128, 128, 128], [255, 0, 0], [0, 255, 0], [0, 0, 255], [255, 255, 0],
            [0, 255, 255], [255, 0, 255], [1, 0, 0], [0, 1, 0], [254, 255, 255], [1, 1, 2], [127, 128, 127]]


@pytest.mark.parametrize("strength", [0.0, 1e-42, 1e-30, 0.4, 1.0])
@pytest.mark.parametrize("gw,gh,tw,th", [
    (1, 1, 1, 1), (300, 2, 1, 3), (7, 5, 2, 1), (90, 3, 3, 2), (64, 2, 4, 4), (65, 2, 5, 3), (51, 3, 6, 5),
    (37, 3, 7, 2), (33, 2, 8, 7), (29, 2, 9, 9), (70, 3, 15, 2), (64, 3, 16, 3), (70, 2, 17, 2)])
def test_quads(ctx, orc, gw, gh, tw, th, strength):
    rng = np.random.default_rng(gw * 131 + tw)
    mats = np.empty((40, th + 3, tw + 2, 3), np.uint8)
    for k in range(40):
        base = np.array(EXTREMES[k]) if k < len(EXTREMES) else rng.integers(0, 256, 3)
        noise = rng.integers(-30, 31, mats.shape[1:]) if k % 3 == 0 else 0
        mats[k] = np.clip(base + noise, 0, 255)
    target = rng.integers(0, 256, (gh * th, gw * tw, 3)).astype(np.uint8)
    target[: gh * th // 2] = 200  # cells that want no hue
    grid = rng.integers(0, len(mats), gw * gh).astype(np.int32)
    grid[rng.random(gw * gh) < 0.1] = -1
    lib = ctx.library_from_pixels(mats)
    got = ctx.composite(lib, target, grid, gw, gh, strength)
    lib.close()
    np.testing.assert_array_equal(got, orc.composite(target, mats, grid, gw, gh, strength))
