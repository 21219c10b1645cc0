"""Annealing that begins cold on small grids (k_anneal.hip).

Whole blocks of proposals and rounds that expect acceptance both pay only while
most proposals are accepted, so a run that rejects most must soon be in rounds
that expect none, and stay there.  How many of those a run takes follows from
the one-at-a-time chain's decisions: a round ends at the first proposal one of
whose ten cells (its two and their neighbours) a swap accepted earlier in the
round has changed.  The device may take 8% more and 8, for the blocks and rounds
that find out.  Results equal the oracle's bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rounds(orc, accept, gw, gh, n, seed):
    """Rounds that expect no acceptance, for the given decisions."""
    def cells(it):
        x1, y1, x2, y2 = (orc.draw(seed, it, k) * b >> 32 for k, b in enumerate((gw, gh, gw, gh)))
        return (x1, y1), (x2, y2)
    prop = [cells(it) for it in range(n)]
    s = rounds = 0
    while s < n:
        changed, end = set(), min(s + 64, n)
        for it in range(s, end):
            a, b = prop[it]
            if a == b:
                continue
            near = {(x + dx, y + dy) for x, y in (a, b) for dx, dy in ((0, 0), (1, 0), (-1, 0), (0, 1), (0, -1))}
            if near & changed:
                end = it
                break
            if accept[it]:
                changed |= {a, b}
        s = end
        rounds += 1
    return rounds


@pytest.mark.parametrize("t0", [0.02, 0.005, 1e-6])
@pytest.mark.parametrize("gw,gh,n", [(8, 6, 100), (20, 15, 300), (50, 28, 500)])
def test_cold_runs(ctx, orc, gw, gh, n, t0):
    rng = np.random.default_rng(gw)
    lab = (rng.random((n, 3)) * [100, 60, 60] - [0, 30, 30]).astype(np.float32)
    grid = rng.integers(0, n, gw * gh).astype(np.int32)
    its = 4000
    want = orc.anneal(lab, grid, gw, gh, its, t0, 0.99995, seed=3, trace=True)
    lib = ctx.library_from_lab(lab)
    got = ctx.anneal(lib, grid, gw, gh, its, t0, 0.99995, seed=3)
    lib.close()
    np.testing.assert_array_equal(got["grid"], want["grid"])
    for k in ("initial_cost", "final_cost", "best_cost"):
        assert np.float32(got["result"][k]) == np.float32(want["result"][k])
    assert got["result"]["accepted_count"] == want["result"]["accepted_count"]
    assert np.mean(want["trace_accept"]) < 0.5
    expected = _rounds(orc, want["trace_accept"], gw, gh, its, 3)
    assert got["result"]["rounds"] <= 1.08 * expected + 8, (got["result"]["rounds"], expected)
