"""TiledCopy plans that give each thread two words: inputs of 16 to 104 MiB with
rows of at least 64 bytes. The plan at both ends of that range, and the kernel's
per-thread code replayed on the host at tensors that end inside a workgroup's
second word, with outputs that start anywhere in a line."""
import ctypes

import numpy as np
import pytest

import librett_amd as L
import oracle
from librett_amd import data
from oracle import counters as OC
from test_kernel_edges_cpu import at_phase


def copies(dim, perm, elem):
    return [(i, c) for i, c in enumerate(L.host_candidates(dim, perm, elem)) if c["method"] == L.TILED_COPY]


@pytest.mark.parametrize("dim,elem,words", [
    ([16, 512, 511], 4, 1), ([16, 512, 513], 4, 2), ([16, 1305, 1305], 4, 2), ([16, 1306, 1306], 4, 1),
    ([15, 700, 700], 4, 1), ([8, 512, 513], 8, 2), ([7, 700, 700], 8, 1), ([4, 512, 513], 16, 2), ([3, 700, 700], 16, 1),
    ([2048, 50, 40], 8, 2), ([2048, 84, 84], 8, 1),
])
def test_words_per_thread(dim, elem, words):
    got = copies(dim, [0, 2, 1], elem)
    per = 256 * (16 // elem) * words
    assert got and all(c["feat"][2] == -(-int(np.prod(dim)) // per) for _, c in got)


# 16 MiB and a little more: the last workgroup holds less than its first word
# per thread, between one and two, and a cut word.
@pytest.mark.parametrize("dim,elem", [
    ([16, 1025, 257], 4), ([33, 367, 349], 4), ([1031, 64, 65], 4), ([9, 500, 479], 8), ([2053, 32, 33], 8),
    ([5, 461, 459], 16), ([1027, 31, 33], 16),
])
def test_two_words_per_thread_replayed(dim, elem):
    perm = [0, 2, 1]
    n = int(np.prod(dim))
    assert n * elem >= 16 << 20
    x = data.uniform(n, elem, 47)
    ref = oracle.transpose(dim, perm, elem, x).view(np.uint8)
    args = (3, L._iarr(dim), L._iarr(perm), elem, ctypes.byref(L.mi355x_desc()))
    line = 128 // elem
    for k in (0, 1, line - 1):
        src, dst = at_phase(n, x.dtype, (3 * k) % line), at_phase(n, x.dtype, k)
        src[:] = x
        for i, c in copies(dim, perm, elem):
            dst[:] = 7
            assert L.lib().librett_c_host_replay(*args, i, src.ctypes.data, dst.ctypes.data) == L.LIBRETT_SUCCESS
            assert np.array_equal(dst.view(np.uint8), ref), (dim, elem, k, c["desc"])


@pytest.mark.parametrize("dim,elem", [([33, 367, 349], 4), ([4, 513, 512], 16)])
def test_two_words_per_thread_counted(dim, elem):
    n = int(np.prod(dim)) * elem
    for i, c in copies(dim, [0, 2, 1], elem):
        got = L.host_candidate_counters(dim, [0, 2, 1], elem, i)
        assert got["ld_bytes"] == got["st_bytes"] == n, c["desc"]
        kern = L.host_access_trace(dim, [0, 2, 1], elem, i, 1)
        mine = L.host_access_trace(dim, [0, 2, 1], elem, i, 0)
        order = [np.lexsort((r[:, 2], r[:, 3], r[:, 1], r[:, 0])) for r in (kern, mine)]
        assert np.array_equal(kern[order[0]][:, [0, 1, 3, 4, 5]], mine[order[1]][:, [0, 1, 3, 4, 5]]), c["desc"]
        for k, v in OC.counts(kern).items():
            assert got[k] == v, (c["desc"], k, got[k], v)


@pytest.mark.parametrize("dim,perm,elem", [([2, 61, 67], [0, 2, 1], 4), ([3, 7, 9, 40], [0, 3, 1, 2], 4), ([2, 90, 45], [0, 2, 1], 8)])
def test_lines_of_many_row_pieces(dim, perm, elem):
    # Up to 512 pieces of rows in one item, scattered over the input: the
    # counters sort them, and count what the model counts where it walks every item.
    for i, c in copies(dim, perm, elem):
        assert 1 < c["feat"][2] <= 24
        got = L.host_candidate_counters(dim, perm, elem, i)
        assert (got["read_lines"], got["write_lines"], got["partial_lines"]) == (
            c["read_lines"], c["write_lines"], c["partial_lines"]), c["desc"]
