"""Host copies around the sizes from which they are staged (mh_stage.hip).

One buffer up is staged from 24 MiB, one down from 6 MiB; gathered images are
staged at any size, by one thread below 5 MiB and by three from there, in chunks
of 1 to 4 MiB.  The totals stand just under, at and just over these sizes, at a
whole number of chunks and with a last chunk of a few bytes.  Everything
compared is equal bit for bit: each cell's, image's or material's own value
from the oracle, and a matrix whose entries name their place.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@pytest.mark.parametrize("extra", [-3072, 0, 3072, 4 * MIB + 3072])
def test_one_buffer_up(ctx, orc, extra):
    rng = np.random.default_rng(24)
    rows = (24 * MIB + extra) // 3072
    img = rng.integers(0, 256, (rows, 1024, 3), dtype=np.uint8)
    gw, gh = 16, 64
    got = ctx.cell_lab_means(img, gw, gh).reshape(gh, gw, 3)
    th = rows // gh
    cells = [(0, 0), (gw - 1, 0), (3, gh // 2), (0, gh - 1), (gw - 1, gh - 1)]
    for x, y in cells:
        one = np.ascontiguousarray(img[y * th:(y + 1) * th, x * 64:(x + 1) * 64])
        want = orc.stack_lab_means(one[None])[0]
        np.testing.assert_array_equal(got[y, x].view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("count", [2047, 2048, 2049, 2731])
def test_library_pixels_up(ctx, orc, count):
    """12 KiB a material: around 24 MiB, and 32 MiB and a little."""
    rng = np.random.default_rng(count)
    px = rng.integers(0, 256, (count, 64, 64, 3), dtype=np.uint8)
    lib = ctx.library_from_pixels(px)
    got = lib.lab()
    lib.close()
    want = orc.stack_lab_means(px)
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("n", [1254, 1255, 2048, 2049, 3000])
def test_one_buffer_down(ctx, orc, n):
    """n x n floats: 1 KiB under and 9 KiB over 6 MiB, 16 MiB, a row more, 34 MiB."""
    rng = np.random.default_rng(n)
    lab = (rng.random((n, 3)) * [100, 60, 60]).astype(np.float32)
    lib = ctx.library_from_lab(lab)
    lib.build_similarities()
    full, packed = lib.similarities(), lib.similarities(packed=True)
    lib.close()
    d = lab[:, None, :] - lab[None, :, :]
    want = np.sqrt(d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1] + d[..., 2] * d[..., 2])
    np.testing.assert_array_equal(full.view(np.uint32), want.view(np.uint32))
    np.testing.assert_array_equal(packed.view(np.uint32), want[np.triu_indices(n, 1)].view(np.uint32))


@pytest.mark.parametrize("sizes", [
    [(64, 16)] * 341 + [(1, 341)],               # 1 MiB - 1
    [(64, 16)] * 341 + [(64, 5), (1, 22)],       # 1 MiB + 2
    [(512, 512)] * 6 + [(100, 1000)],            # 4.8 MiB, one thread
    [(512, 512)] * 6 + [(512, 683)],             # 5.5 MiB, three threads
    [(8, 8)] * 2500 + [(640, 640)],
])
def test_gathered(ctx, orc, sizes):
    rng = np.random.default_rng(len(sizes))
    images = [rng.integers(0, 256, (h, w, 3), dtype=np.uint8) for h, w in sizes]
    want = np.stack([orc.stack_lab_means(im[None])[0] for im in images])
    got = ctx.average_lab_many(images)
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    lib = ctx.library_from_images(images)
    np.testing.assert_array_equal(lib.lab().view(np.uint32), want.view(np.uint32))
    lib.close()
