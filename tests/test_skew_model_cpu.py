"""The model's line counts of skewed tiles, against the access counters' own
walk of every item: all columns of a tile on one line offset, every offset
between lines, a tile of 64 columns, of one column, and planes over dim groups.
Plans of at most 24 items, which the model walks whole."""
import pytest

import librett_amd as L


@pytest.mark.parametrize("dim,perm", [
    ([64, 161], [1, 0]), ([65, 129], [1, 0]), ([64, 3, 131], [2, 1, 0]), ([33, 257], [1, 0]), ([7, 9, 140], [2, 0, 1]),
    ([64, 13, 17], [1, 2, 0]), ([5, 30, 133], [2, 1, 0]),
])
@pytest.mark.parametrize("elem", [4, 8, 16])
def test_modelled_lines_of_skewed_tiles(dim, perm, elem):
    seen = 0
    for i, c in enumerate(L.host_candidates(dim, perm, elem)):
        if " skew" not in c["desc"] or c["feat"][2] > 24:
            continue
        got = L.host_candidate_counters(dim, perm, elem, i)
        assert (got["read_lines"], got["write_lines"], got["partial_lines"]) == (
            c["read_lines"], c["write_lines"], c["partial_lines"]), c["desc"]
        seen += 1
    assert seen


@pytest.mark.parametrize("dim,elem,packed", [([32, 40, 50], 4, False), ([31, 40, 50], 4, True), ([16, 40, 50], 8, False),
                                             ([8, 40, 50], 16, False), ([7, 40, 50], 16, True)])
def test_batched_rows_of_whole_lines_have_only_the_copy(dim, elem, packed):
    # Rows of 128 bytes and more are copied in the batched engine; shorter ones
    # keep their Packed plans. Each plan gives the oracle's output.
    import ctypes

    import numpy as np

    import oracle
    from librett_amd import data
    perm, n = [0, 2, 1], int(np.prod(dim))
    x = data.uniform(n, elem, 5)
    ref = oracle.transpose(dim, perm, elem, x).view(np.uint8)
    count = ctypes.c_int()
    args = (3, L._iarr(dim), L._iarr(perm), elem, ctypes.byref(L.mi355x_desc()))
    assert L.lib().librett_c_batch_host_candidate(*args, 0, 0, 0, 0, None, None, ctypes.byref(count)) == L.LIBRETT_SUCCESS
    assert (count.value > 1) == packed
    for i in range(count.value):
        out = np.zeros_like(x)
        assert L.lib().librett_c_batch_host_candidate(*args, i, 0, 0, 0, x.ctypes.data, out.ctypes.data,
                                                      None) == L.LIBRETT_SUCCESS
        assert np.array_equal(out.view(np.uint8), ref)
