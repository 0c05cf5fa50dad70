"""The kernels' per-thread code at the sizes where it can go wrong, replayed on
the host with inputs and outputs that start anywhere in a cache line: every
candidate plan and every batch-mode candidate, bit for bit against the
oracle, between guard bands."""
import ctypes

import numpy as np
import pytest

import librett_amd as L
import oracle
from librett_amd import data


def at_phase(n, dtype, k):
    """An array of n elements that starts k elements into a cache line."""
    line = 128 // dtype.itemsize
    a = np.zeros(n + 2 * line, dtype=dtype)
    s = (-a.ctypes.data // dtype.itemsize) % line + k
    return a[s:s + n]


def replay_all(dim, perm, elem, phases, methods=None):
    n = int(np.prod(dim))
    x = data.uniform(n, elem, 43)
    ref = oracle.transpose(dim, perm, elem, x).view(np.uint8)
    args = (len(dim), L._iarr(dim), L._iarr(perm), elem, ctypes.byref(L.mi355x_desc()))
    ran = 0
    for k in phases:
        src, dst = at_phase(n, x.dtype, (3 * k) % (128 // elem)), at_phase(n, x.dtype, k)
        src[:] = x
        for i, c in enumerate(L.host_candidates(dim, perm, elem)):
            if methods and c["method"] not in methods:
                continue
            dst[:] = 7
            r = L.lib().librett_c_host_replay(*args, i, src.ctypes.data, dst.ctypes.data)
            assert r == L.LIBRETT_SUCCESS and np.array_equal(dst.view(np.uint8), ref), (dim, perm, elem, k, c["desc"])
            ran += 1
        m = ctypes.c_int(0)
        for i in range(L.batch_host_candidates(dim, perm, elem)):
            for fallback in (0, 1):
                dst[:] = 7
                r = L.lib().librett_c_batch_host_candidate(*args, i, fallback, 32 << 10, 11, src.ctypes.data,
                                                           dst.ctypes.data, ctypes.byref(m))
                assert r == L.LIBRETT_SUCCESS and np.array_equal(dst.view(np.uint8), ref), (dim, perm, elem, k, i)
                ran += 1
    return ran


@pytest.mark.parametrize("elem", [4, 8, 16])
@pytest.mark.parametrize("dim,perm", [
    ([2, 3, 5], [0, 2, 1]), ([3, 7, 11, 2], [0, 3, 2, 1]), ([33, 5, 7, 4, 3], [0, 4, 2, 3, 1]),
    ([1031, 3, 5], [0, 2, 1]), ([4097, 2, 3], [0, 2, 1]), ([613], [0]), ([1], [0]),
])
def test_copy_rows(dim, perm, elem):
    assert replay_all(dim, perm, elem, [0, 1, 128 // elem - 1], methods=(L.TRIVIAL, L.TILED_COPY)) > 0


SKEWED = [([65, 129], [1, 0], 4), ([33, 259, 5], [1, 2, 0], 4), ([5, 29, 7, 67], [3, 1, 0, 2], 8),
          ([65, 129], [1, 0], 8), ([17, 33], [1, 0], 16), ([9, 11, 35], [2, 1, 0], 16)]
# Narrow planes, 1 to 12 columns, and the same the other way round (short
# columns): one tile and several, cut by the plane's end, with outer dims that
# move the phase.
NARROW = [([7, 1483], [1, 0], 4), ([2, 4099], [1, 0], 4), ([12, 257, 3], [1, 0, 2], 4), ([11, 130, 3], [1, 2, 0], 4),
          ([5, 1100], [1, 0], 8), ([8, 67, 5], [1, 0, 2], 8), ([12, 64, 3], [1, 0, 2], 8),
          ([3, 2051], [1, 0], 16), ([12, 33, 4], [1, 0, 2], 16)]
SHORT = [([1483, 7], [1, 0], 4), ([512, 4, 3], [1, 0, 2], 4), ([4096, 2], [1, 0], 8), ([4099, 2], [1, 0], 4), ([257, 3, 12], [2, 0, 1], 4), ([130, 2, 5, 3], [2, 1, 0, 3], 4),
         ([1100, 5], [1, 0], 8), ([67, 8, 5], [1, 0, 2], 8), ([515, 2, 3], [2, 1, 0], 8),
         ([2051, 3], [1, 0], 16), ([33, 4, 12], [2, 0, 1], 16)]
SKEWED += NARROW + SHORT


@pytest.mark.parametrize("dim,perm,elem", SKEWED)
def test_skewed_tiles(dim, perm, elem):
    # The planner offers skewed tiles for these, and every plan is exact
    # wherever the output starts in a line.
    form = " narrow" if (dim, perm, elem) in NARROW else " short" if (dim, perm, elem) in SHORT else " skew"
    assert any(form in c["desc"] for c in L.host_candidates(dim, perm, elem))
    assert replay_all(dim, perm, elem, [0, 1, 128 // elem - 1]) > 0


@pytest.mark.parametrize("dim,perm,elem", SKEWED)
def test_skewed_tiles_count(dim, perm, elem):
    # Each byte loaded and stored once; the counters' enumeration is what the
    # kernel does; where the model walks every tile, its lines are exact.
    from oracle import counters as OC
    n = int(np.prod(dim)) * elem
    for i, c in enumerate(L.host_candidates(dim, perm, elem)):
        if not any(f in c["desc"] for f in (" skew", " narrow", " short")):
            continue
        got = L.host_candidate_counters(dim, perm, elem, i)
        assert got["ld_bytes"] == got["st_bytes"] == n, c["desc"]
        kern = L.host_access_trace(dim, perm, elem, i, 1)
        mine = L.host_access_trace(dim, perm, elem, i, 0)
        order = [np.lexsort((r[:, 2], r[:, 3], r[:, 1], r[:, 0])) for r in (kern, mine)]
        assert np.array_equal(kern[order[0]][:, [0, 1, 3, 4, 5]], mine[order[1]][:, [0, 1, 3, 4, 5]]), c["desc"]
        for k, v in OC.counts(kern).items():
            if k != "items":  # a tile past every column's end moves nothing
                assert got[k] == v, (c["desc"], k, got[k], v)
        if c["feat"][2] <= 24:
            assert (got["read_lines"], got["write_lines"], got["partial_lines"]) == (
                c["read_lines"], c["write_lines"], c["partial_lines"]), c["desc"]
