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
