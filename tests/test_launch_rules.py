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
