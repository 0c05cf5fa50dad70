"""Kernels at the sizes where they can go wrong, on the GPU: rows and tiles
cut by the tensor's end, outputs that start anywhere in a cache line, the
smallest and a large volume. Every candidate plan, bit for bit against the
oracle, with guard bytes around the output."""
import numpy as np
import pytest

import librett_amd as L
import oracle
from librett_amd import data, hip

pytestmark = pytest.mark.gpu

GUARD = 256


def check(stream, dim, perm, elem, offsets, methods=None, only=None):
    """Every candidate of `methods` on buffers `offset` elements into an allocation."""
    n = int(np.prod(dim))
    x = data.uniform(n, elem, 41)
    ref = oracle.transpose(dim, perm, elem, x).view(np.uint8)
    room = (max(offsets) + n) * elem + 2 * GUARD
    a, b = hip.DeviceBuffer(room), hip.DeviceBuffer(room)
    ran = 0
    try:
        for i, c in enumerate(L.candidates(dim, perm, elem)):
            if methods and c["method"] not in methods or only and only not in c["desc"]:
                continue
            r, h = L.plan_candidate(len(dim), dim, perm, elem, stream, i)
            assert r == L.LIBRETT_SUCCESS, c["desc"]
            for off in offsets:
                print("case:", dim, perm, elem, "offset", off, c["desc"], flush=True)
                at = GUARD + off * elem
                hip.htod(a.ptr + at, x)
                hip.memset(b.ptr, 0xEE, room)
                assert L.librettExecute(h, a.ptr + at, b.ptr + at) == L.LIBRETT_SUCCESS
                hip.stream_sync(stream)
                got = np.empty(room, dtype=np.uint8)
                hip.dtoh(got, b.ptr)
                assert np.array_equal(got[at:at + n * elem], ref), (dim, perm, elem, off, c["desc"])
                assert np.all(got[:at] == 0xEE) and np.all(got[at + n * elem:] == 0xEE), (off, c["desc"])
                ran += 1
            L.librettDestroy(h)
    finally:
        a.free()
        b.free()
    return ran


# Rows shorter than a word, of one word, odd, longer than a workgroup's
# block; volumes that end inside a word; ranks that need several digits.
@pytest.mark.parametrize("elem", [4, 8, 16])
@pytest.mark.parametrize("dim,perm", [
    ([2, 3, 5], [0, 2, 1]), ([3, 7, 11, 2], [0, 3, 2, 1]), ([4, 9, 8], [0, 2, 1]), ([33, 5, 7, 4, 3], [0, 4, 2, 3, 1]),
    ([1031, 3, 5], [0, 2, 1]), ([4097, 2, 3], [0, 2, 1]), ([2, 2, 2, 3, 2, 5, 2, 3], [0, 7, 2, 5, 4, 3, 6, 1]),
])
def test_copy_rows(gpu_stream, dim, perm, elem):
    assert check(gpu_stream, dim, perm, elem, [0, 1, 5, 128 // elem - 1], methods=(L.TILED_COPY,)) >= 4


# Skewed tiles: columns of just enough whole lines, cut tiles on both sides,
# planes over dim groups and outer dims that move the phase, and every place
# in a line that the output can start at.
SKEWED = [([65, 129], [1, 0], 4), ([70, 131, 3], [1, 0, 2], 4), ([33, 259, 5], [1, 2, 0], 4),
          ([5, 29, 7, 67], [3, 1, 0, 2], 8), ([65, 129], [1, 0], 8), ([3, 97, 21], [1, 2, 0], 8),
          ([17, 33], [1, 0], 16), ([7, 67, 5], [1, 0, 2], 16), ([9, 11, 35], [2, 1, 0], 16)]


@pytest.mark.parametrize("dim,perm,elem", SKEWED)
def test_skewed_tiles(gpu_stream, dim, perm, elem):
    line = 128 // elem
    assert check(gpu_stream, dim, perm, elem, [0, 1, line // 2, line - 1], only=" skew") >= 8


# Narrow planes, 1 to 12 columns, and the same the other way round (short
# columns): one tile and several, cut by the plane's end, with outer dims that
# move the phase.
NARROW = [([7, 1483], [1, 0], 4), ([2, 4099], [1, 0], 4), ([12, 257, 3], [1, 0, 2], 4), ([11, 130, 3], [1, 2, 0], 4),
          ([5, 1100], [1, 0], 8), ([8, 67, 5], [1, 0, 2], 8), ([12, 64, 3], [1, 0, 2], 8),
          ([3, 2051], [1, 0], 16), ([12, 33, 4], [1, 0, 2], 16)]
SHORT = [([1483, 7], [1, 0], 4), ([512, 4, 3], [1, 0, 2], 4), ([4096, 2], [1, 0], 8), ([4099, 2], [1, 0], 4), ([257, 3, 12], [2, 0, 1], 4), ([130, 2, 5, 3], [2, 1, 0, 3], 4),
         ([1100, 5], [1, 0], 8), ([67, 8, 5], [1, 0, 2], 8), ([515, 2, 3], [2, 1, 0], 8),
         ([2051, 3], [1, 0], 16), ([33, 4, 12], [2, 0, 1], 16)]


@pytest.mark.parametrize("dim,perm,elem", NARROW + SHORT)
def test_narrow_planes(gpu_stream, dim, perm, elem):
    line = 128 // elem
    form = " narrow" if (dim, perm, elem) in NARROW else " short"
    assert check(gpu_stream, dim, perm, elem, [0, 1, line - 1], only=form) >= 3


@pytest.mark.parametrize("dim, perm", [
    ([33, 2, 3, 2, 3, 35], [5, 4, 3, 2, 1, 0]),
    ([33, 2, 3, 2, 3, 2, 35], [6, 5, 4, 3, 2, 1, 0]),
    ([9, 2, 3, 2, 3], [0, 4, 3, 2, 1]),
    ([9, 2, 3, 2, 3, 2], [0, 5, 4, 3, 2, 1]),
    ([3, 5, 3, 2, 3, 2, 3, 70], [7, 6, 5, 4, 3, 2, 1, 0]),
], ids=["plane, 4 outer dims", "plane, 5", "rows, 4", "rows, 5", "groups, 4 to 6"])
@pytest.mark.parametrize("elem", [4, 8, 16])
def test_outer_dims_around_the_short_arguments(gpu_stream, dim, perm, elem):
    check(gpu_stream, dim, perm, elem, [0, 1], methods=(4, 5))


# Inputs of 104 MiB and more that are read in whole lines: non-temporal loads,
# over planes of one dim and of dim groups (whole tiles and cut ones), and rows.
@pytest.mark.parametrize("dim,perm,elem", [
    ([64, 6, 344, 212], [2, 1, 0, 3], 4), ([32, 12, 344, 106], [2, 1, 0, 3], 8), ([16, 100, 16, 275], [3, 2, 1, 0], 16),
    ([1024, 160, 172], [0, 2, 1], 4),
])
def test_streamed_loads(gpu_stream, dim, perm, elem):
    want = [c["desc"] for c in L.candidates(dim, perm, elem) if c["desc"].endswith(" stream")]
    assert len(want) >= 2 and (perm[0] == 0 or any("groups" in d for d in want))
    assert check(gpu_stream, dim, perm, elem, [0], only=" stream") == len(want)


# 16 to 104 MiB: two words per thread.
@pytest.mark.parametrize("dim,elem", [([33, 367, 349], 4), ([2053, 32, 33], 8), ([5, 461, 459], 16), ([16, 968, 969], 4)])
def test_copy_rows_two_words(gpu_stream, dim, elem):
    assert check(gpu_stream, dim, [0, 2, 1], elem, [0, 1, 128 // elem - 1], methods=(L.TILED_COPY,)) == 6


# More tiles than a row of workgroups holds, in both tile orders, every plan.
@pytest.mark.parametrize("elem", [4, 8, 16])
def test_tiles_of_several_grid_rows(gpu_stream, elem):
    dim, perm = [2, 1100000, 2], [2, 1, 0]
    many = [c["desc"] for c in L.candidates(dim, perm, elem) if c["grid_y"] > 1 and c["method"] == L.TILED]
    assert many and any(d.endswith(" xcd") for d in many) and any(not d.endswith(" xcd") for d in many)
    assert check(gpu_stream, dim, perm, elem, [0], only=" grid 1048576x2") == len(many)


# On both sides of the short kernel arguments' four outer dims: plans of either
# kernel, which test_outer_dims_around_the_short_arguments runs, are there.
@pytest.mark.parametrize("dim,perm,outer,kind", [
    ([33, 2, 3, 2, 3, 35], [5, 4, 3, 2, 1, 0], 4, "Tiled"), ([33, 2, 3, 2, 3, 2, 35], [6, 5, 4, 3, 2, 1, 0], 5, "Tiled"),
    ([9, 2, 3, 2, 3], [0, 4, 3, 2, 1], 4, "TiledCopy"), ([9, 2, 3, 2, 3, 2], [0, 5, 4, 3, 2, 1], 5, "TiledCopy"),
])
@pytest.mark.parametrize("elem", [4, 8, 16])
def test_both_sides_of_the_short_arguments_run(gpu_stream, dim, perm, outer, kind, elem):
    # Planes of one dim each leave all but two of the dims outside; rows all but one.
    assert len(dim) - (2 if kind == "Tiled" else 1) == outer
    ran = check(gpu_stream, dim, perm, elem, [0, 1], methods=(L.TILED if kind == "Tiled" else L.TILED_COPY,))
    plain = [c for c in L.candidates(dim, perm, elem) if c["desc"].startswith(kind + " ") and "groups" not in c["desc"]]
    assert len(plain) >= 2 and ran >= 2 * len(plain)
