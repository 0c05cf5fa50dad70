"""Batches whose problem count sits at the edges of the 64-way search for a
unit's problem: one, two and three steps, full and just past full. Problems of
one unit, so that every problem is some unit's first."""
import numpy as np
import pytest

import librett_amd as L
from librett_amd import hip
from test_gpu_batch import Slab

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 2, 63, 64, 65, 127, 128, 129, 4095, 4096, 4097])
def test_unit_finds_its_problem(gpu_stream, count):
    print("case:", count, "problems", flush=True)
    rng = np.random.default_rng(count)
    probs = [([int(rng.integers(2, 6)), int(rng.integers(2, 6))], [1, 0], 8) for _ in range(count)]
    slab = Slab(probs)
    b = L.Batch(probs, gpu_stream, tune=0)
    try:
        b.set_buffers(slab.in_ptrs(), slab.out_ptrs())
        assert b.execute(use_graph=False) == L.LIBRETT_SUCCESS
        hip.stream_sync(gpu_stream)
        assert slab.check() == []
    finally:
        b.destroy()
        slab.free()


def test_units_of_several_grid_rows(gpu_stream):
    # One 17 GB problem of 1 048 832 units, 256 more than a row of workgroups
    # holds: filled and checked on the device.
    dim, perm, elem = [64, 4097, 4096], [0, 2, 1], 16
    n = int(np.prod(dim, dtype=np.int64)) * elem
    print("case:", dim, perm, elem, flush=True)
    a, c = hip.DeviceBuffer(n), hip.DeviceBuffer(n)
    b = L.Batch([(dim, perm, elem)], gpu_stream, tune=0)
    try:
        assert b.info()["total_units"] > 1 << 20
        L.check_fill(a.ptr, n, gpu_stream)
        hip.memset(c.ptr, 0, n)
        b.set_buffers([a.ptr], [c.ptr])
        assert b.execute(use_graph=False) == L.LIBRETT_SUCCESS
        hip.stream_sync(gpu_stream)
        assert L.check_transpose(c.ptr, dim, perm, elem, gpu_stream) == (0, -1)
    finally:
        b.destroy()
        a.free()
        c.free()
