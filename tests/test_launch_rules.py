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


@pytest.mark.parametrize("chunk", [1, 3, 32, 299, 300, 301, 2**32 - 1])
@pytest.mark.parametrize("lead", [0, 5])
def test_schedule_of_one_range(chunk, lead):
    """Every entry against the definition: pieces of `chunk` edges and one rest, by length, then the whole rows by
    length; slots and split rows by row; lengths at the piece length and its multiples, empty rows, edges before the
    first row, a piece length beyond every row and one that no array could hold a count for."""
    deg = np.concatenate([[300, 0, 299, 301, 600, 1, 32, 64, 0, 33], np.random.default_rng(9).integers(0, 301, 40)])
    co = np.zeros(deg.size + 1, dtype=np.uint32)
    co[1:] = np.cumsum(deg)
    co += np.uint32(lead)
    items, n_splits, n_partials = schedule(co, None, 0, chunk, 0)
    pieces, whole = [], []
    for r in range(deg.size):
        b, e = int(co[r]), int(co[r + 1])
        if e - b <= chunk:
            whole.append((r, b, e, int(NO_SLOT)))
        else:
            pieces += [(r, k, min(e, k + chunk), len(pieces) + j) for j, k in enumerate(range(b, e, chunk))]
    want = sorted(pieces, key=lambda p: p[1] - p[2]) + sorted(whole, key=lambda p: p[1] - p[2])
    assert n_splits == int((deg > chunk).sum()) and n_partials == len(pieces)
    assert np.array_equal(items, np.array(want, dtype=np.uint32))
