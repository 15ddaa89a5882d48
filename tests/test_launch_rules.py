"""Sizes that the library picks by itself, checked without a GPU."""
import numpy as np
import pytest

from test_plan_schedule import NO_SLOT, schedule


@pytest.mark.parametrize("edges,longest", [(1000, 32), (10556, 32), (64 * 8192 - 1, 32), (64 * 8192, 64), (2480000, 256),
                                           (33554431, 2048), (33554432, 4096)])
def test_default_piece_length_follows_the_edge_count(edges, longest):
    """One row above the piece length, the remaining edges in rows below it."""
    short = np.full(max(1, (edges - longest - 1) // 30), 30)
    deg = np.concatenate([short, [longest + 1, edges - longest - 1 - int(short.sum())]])
    co = np.zeros(deg.size + 1, dtype=np.uint32)
    co[1:] = np.cumsum(deg)
    items, n_splits, n_partials = schedule(co, None, 0, 0, 0)
    assert n_splits == 1 and n_partials == 2
    pieces = items[items[:, 3] != NO_SLOT]
    assert sorted((pieces[:, 2] - pieces[:, 1]).tolist()) == [1, longest]


def test_root_of_a_degree_in_32_bits():
    """The weights' roots: for every degree a float can hold, the 32-bit root is the 64-bit one rounded."""
    deg = np.concatenate([np.arange(1, 1 << 20), np.arange((1 << 24) - (1 << 16), 1 << 24),
                          np.random.default_rng(1).integers(1, 1 << 24, 1 << 20)]).astype(np.uint32)
    assert np.array_equal(np.sqrt(deg.astype(np.float32)), np.sqrt(deg.astype(np.float64)).astype(np.float32))


@pytest.mark.parametrize("chunk", [1, 7, 64, 100000])
def test_pieces_of_one_range_are_issued_by_length(chunk):
    """Longest first, pieces of equal length in the order of their slots; the whole rows behind them likewise by row."""
    deg = np.random.default_rng(chunk).integers(0, 300, 500)
    co = np.zeros(deg.size + 1, dtype=np.uint32)
    co[1:] = np.cumsum(deg)
    items, n_splits, n_partials = schedule(co, None, 0, chunk, 0)
    n = items[:, 2].astype(np.int64) - items[:, 1]
    assert n_splits == int((deg > chunk).sum()) and n_partials == int((items[:, 3] != NO_SLOT).sum())
    for part, key in ((slice(0, n_partials), 3), (slice(n_partials, None), 0)):
        order = np.lexsort((items[part, key], -n[part]))
        assert np.array_equal(order, np.arange(order.size))
    assert int(n.sum()) == int(co[-1])
