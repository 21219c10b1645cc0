"""Annealing in whole blocks of 64 proposals (k_anneal.hip), against the oracle.

The cases stand where a block's chain of cells, its end or the change to rounds
can go wrong: proposal counts around one and two blocks and the ring of 256
draws, grids of so few cells that every swap meets the ones before (the longest
chains) and of one row or column, the largest grid taken (4,096 cells) and the
next, Labs in LDS and in memory, and too many for both them and the blocks'
tables, ids of 16 and 32 bits, empty cells, equal materials, and temperatures
that reject one proposal in a few blocks, one in a few proposals, and most.
Everything equals the one-at-a-time chain bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # gw, gh, n, distinct Labs, empty share, proposals, t0, decay
    (1, 1, 2, 2, 0.0, 70, 100.0, 0.99995),
    (2, 1, 2, 2, 0.0, 64, 100.0, 0.99995),
    (2, 2, 4, 4, 0.0, 300, 100.0, 0.99995),
    (1, 9, 9, 9, 0.0, 127, 100.0, 0.99995),
    (13, 1, 5, 3, 0.2, 128, 100.0, 0.99995),
    (8, 8, 64, 64, 0.0, 65, 100.0, 0.99995),
    (20, 15, 300, 300, 0.1, 1000, 8.0, 0.9999),
    (31, 17, 500, 9, 0.0, 1500, 1.0, 0.999),
    (24, 18, 10500, 10500, 0.0, 1200, 20.0, 0.9995),
    (24, 18, 33000, 33000, 0.05, 900, 50.0, 0.999),
    (50, 28, 500, 500, 0.0, 3000, 100.0, 0.998),
    (63, 65, 7500, 7500, 0.0, 700, 100.0, 0.99995),
    (64, 64, 1500, 1500, 0.0, 2500, 30.0, 0.9995),
    (64, 64, 1500, 1500, 0.01, 63, 100.0, 0.99995),
    (17, 241, 200, 200, 0.0, 1300, 100.0, 0.99995),
]


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("gw,gh,n,distinct,empty,iters,t0,decay", CASES)
def test_blocks(ctx, orc, gw, gh, n, distinct, empty, iters, t0, decay):
    rng = np.random.default_rng(gw * 977 + n + iters)
    lab = (rng.random((n, 3)) * [100, 60, 60] - [0, 30, 30]).astype(np.float32)
    lab = lab[np.arange(n) % distinct]
    grid = rng.integers(0, n, gw * gh).astype(np.int32)
    grid[rng.random(gw * gh) < empty] = -1
    lib = ctx.library_from_lab(lab)
    got = ctx.anneal(lib, grid, gw, gh, iters, t0, decay, seed=iters + 3, greedy=False, trace=True)
    lib.close()
    want = orc.anneal(lab, grid, gw, gh, iters, t0, decay, seed=iters + 3, greedy=False, trace=True)
    np.testing.assert_array_equal(got["trace_accept"], want["trace_accept"])
    np.testing.assert_array_equal(_bits(got["trace_delta"]), _bits(want["trace_delta"]))
    np.testing.assert_array_equal(got["grid"], want["grid"])
    for key in ("initial_cost", "final_cost", "best_cost"):
        assert _bits(np.float32(got["result"][key])) == _bits(np.float32(want["result"][key])), key
    for key in ("improved_count", "accepted_count", "iterations", "evaluated"):
        assert got["result"][key] == want["result"][key], key
