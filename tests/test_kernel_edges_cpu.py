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
