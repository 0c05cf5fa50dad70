"""Launch grids on the host: a batch's units found by their workgroups, over the
edges of the 64-way search and over grids of several rows, and the tiles of a
plan that needs more than one row of workgroups."""
import ctypes

import numpy as np
import pytest

import librett_amd as L
import oracle
from librett_amd import data


@pytest.mark.parametrize("count", [1, 2, 63, 64, 65, 127, 129, 4095, 4096, 4097])
def test_units_find_their_problem(count):
    rng = np.random.default_rng(count)
    probs = [([int(rng.integers(2, 6)), int(rng.integers(2, 6))], [1, 0], 8) for _ in range(count)]
    xs = [data.uniform(int(np.prod(d)), e, i) for i, (d, p, e) in enumerate(probs)]
    refs = [oracle.transpose(d, p, e, x) for (d, p, e), x in zip(probs, xs)]
    # One row, rows that the units fill, and rows whose last is cut.
    for row in (0, count, 64, 11, 1):
        got = L.batch_host_replay(probs, xs, grid=row)
        assert all(np.array_equal(y, r) for y, r in zip(got, refs)), row


def test_units_of_several_rows():
    # Problems of many units each, of every kernel family.
    probs = [([70, 131, 3], [1, 0, 2], 4), ([33, 5, 70, 4], [0, 2, 1, 3], 8), ([5, 29, 7, 67], [3, 1, 0, 2], 8),
             ([6, 12, 6, 11, 5, 2], [5, 4, 3, 2, 1, 0], 16), ([64, 96, 40], [2, 1, 0], 4), ([9000], [0], 4)]
    xs = [data.uniform(int(np.prod(d)), e, i) for i, (d, p, e) in enumerate(probs)]
    refs = [oracle.transpose(d, p, e, x) for (d, p, e), x in zip(probs, xs)]
    for row in (0, 1, 3, 7, 64):
        got = L.batch_host_replay(probs, xs, grid=row)
        assert all(np.array_equal(y, r) for y, r in zip(got, refs)), row


MANY = ([2, 1100000, 2], [2, 1, 0])


def test_grid_of_several_rows_is_described():
    got = [c for c in L.host_candidates(*MANY, 16) if c["grid_y"] > 1 and c["method"] == L.TILED]
    assert got
    for c in got:
        assert c["grid_x"] == 1 << 20 and c["grid_y"] == 2
        assert " grid 1048576x2" in c["desc"]


@pytest.mark.parametrize("xcd", [False, True])
def test_tiles_of_several_rows(xcd):
    # 1.1 million tiles: the second row of workgroups ends early.
    dim, perm = MANY
    i, c = next((i, c) for i, c in enumerate(L.host_candidates(dim, perm, 16))
                if c["grid_y"] > 1 and "16x16" in c["desc"] and c["desc"].endswith(" xcd") == xcd)
    x = data.uniform(int(np.prod(dim)), 16, 3)
    y = L.host_replay(dim, perm, 16, i, x)
    assert np.array_equal(y.view(np.uint8), oracle.transpose(dim, perm, 16, x).view(np.uint8)), c["desc"]
