"""Annealing rounds and the ordered sums (k_anneal.hip), against the oracle.

The cases stand where a round's prefix or a sum's short cut can go wrong:
proposal counts around a window of 64 and the ring of 256 draws, grids of a
few cells (every proposal meets the one before), stamps one a cell and shared
(above 16,384 cells), ids of 16 and 32 bits, the library's Labs in LDS and
not, temperatures that accept nearly all, about half and nearly none (both
ways to find the prefix, and the change between them), greedy runs, empty
cells, libraries of one material and of few distinct ones (equal terms, which
meet half-way cases and binade edges of the sums together), and grids larger
than a chunk of the initial cost.  Everything equals the one-at-a-time chain
bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # gw, gh, n, distinct Labs, empty share, proposals, t0, decay, greedy
    (2, 2, 4, 4, 0.0, 63, 100.0, 0.99995, False),
    (3, 1, 3, 3, 0.0, 65, 1.0, 0.999, False),
    (5, 7, 1, 1, 0.0, 129, 100.0, 0.99995, False),
    (20, 15, 300, 300, 0.0, 1000, 100.0, 0.99995, False),
    (20, 15, 300, 300, 0.3, 1000, 1.0, 0.995, False),
    (21, 15, 300, 7, 0.05, 700, 0.05, 0.99, False),
    (20, 15, 300, 300, 0.0, 1000, 100.0, 0.99995, True),
    (80, 60, 1500, 1500, 0.0, 3000, 0.5, 0.9995, False),
    (80, 60, 1500, 1500, 0.0, 1, 100.0, 0.99995, False),
    (129, 127, 9000, 9000, 0.0, 2000, 100.0, 0.99995, False),
    (129, 128, 900, 900, 0.02, 4000, 1.0, 0.999, False),
    (201, 119, 6000, 40, 0.0, 3000, 100.0, 0.99, False),
    (160, 120, 33000, 33000, 0.0, 1500, 10.0, 0.999, False),
    (300, 171, 500, 500, 0.01, 3000, 2.0, 0.999, False),
    (300, 171, 500, 500, 0.0, 600, 100.0, 0.99995, True),
]


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("gw,gh,n,distinct,empty,iters,t0,decay,greedy", CASES)
def test_rounds(ctx, orc, gw, gh, n, distinct, empty, iters, t0, decay, greedy):
    rng = np.random.default_rng(gw * 1013 + n + iters)
    lab = (rng.random((n, 3)) * [100, 60, 60] - [0, 30, 30]).astype(np.float32)
    lab = lab[np.arange(n) % distinct]
    grid = rng.integers(0, n, gw * gh).astype(np.int32)
    grid[rng.random(gw * gh) < empty] = -1
    lib = ctx.library_from_lab(lab)
    got = ctx.anneal(lib, grid, gw, gh, iters, t0, decay, seed=iters + 5, greedy=greedy, trace=True)
    assert _bits(np.float32(ctx.total_cost(lib, grid, gw, gh))) == _bits(orc.total_cost(lab, grid, gw, gh))
    lib.close()
    want = orc.anneal(lab, grid, gw, gh, iters, t0, decay, seed=iters + 5, greedy=greedy, trace=True)
    np.testing.assert_array_equal(got["trace_accept"], want["trace_accept"])
    np.testing.assert_array_equal(_bits(got["trace_delta"]), _bits(want["trace_delta"]))
    np.testing.assert_array_equal(got["grid"], want["grid"])
    for key in ("initial_cost", "final_cost", "best_cost"):
        assert _bits(np.float32(got["result"][key])) == _bits(np.float32(want["result"][key])), key
    for key in ("improved_count", "accepted_count", "iterations", "evaluated"):
        assert got["result"][key] == want["result"][key], key
