"""Plans that read their input with non-temporal loads, on the host.

Which plans these are depends on the tensor's size, and LIBRETT_STREAM_MB
moves the line: with 0 the small shapes here take the branches that the
kernels otherwise take for large tensors. The library reads it once, so each
test asks a process of its own. Every plan there, replayed by the kernels' own
per-thread code, must equal the oracle bit for bit."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# Whole input lines: planes of one dim, of several y dims, of several x dims
# and of both, with whole tiles and cut ones; rows.
SHAPES = [([128, 96], [1, 0]), ([128, 130], [1, 0]), ([128, 4, 64], [2, 1, 0]), ([64, 6, 34, 2], [2, 1, 0, 3]),
          ([32, 128, 8, 3], [2, 1, 0, 3]), ([8, 16, 4, 32], [3, 2, 1, 0]), ([64, 5, 7], [0, 2, 1])]

CHILD = """
import json, sys
sys.path[:0] = [%r, %r]
import librett_amd as L
from test_planner_cpu import replay_all
out = []
for dim, perm in json.loads(sys.argv[1]):
    for elem in (4, 8, 16):
        out += [(dim, elem, c["desc"]) for c in replay_all(dim, perm, elem)]
print(json.dumps(out))
""" % (ROOT, os.path.join(ROOT, "tests"))


def plans(megabytes, shapes):
    env = dict(os.environ, LIBRETT_STREAM_MB=str(megabytes))
    r = subprocess.run([sys.executable, "-c", CHILD, json.dumps(shapes)], env=env, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return json.loads(r.stdout.splitlines()[-1])


@pytest.mark.parametrize("dim,perm", SHAPES)
def test_streamed_plans(dim, perm):
    got = plans(0, [(dim, perm)])
    streamed = [d for _, _, d in got if d.endswith(" stream")]
    assert streamed
    if perm[0] == 0:
        assert all(d.startswith("TiledCopy") for d in streamed)
    elif len(dim) > 2:
        # Planes over several dims among them.
        assert any("groups" in d for d in streamed)


def test_small_inputs_are_not_streamed():
    assert not any("stream" in d for _, _, d in plans(96, SHAPES))


@pytest.mark.parametrize("dim,elem,streamed", [
    ([1024, 256, 256], 4, True), ([1024, 96, 250], 4, False), ([2307, 115, 126], 8, False),
    ([2307, 50, 112], 8, False), ([2307, 150, 145], 8, False), ([2307, 150, 146], 8, True), ([129, 700, 700], 8, False),
])
def test_rows_cut_by_lines_stream_only_far_beyond_the_cache(dim, elem, streamed):
    # 256 MiB of whole lines, and 94; cut rows of 18 KB from 384 MiB on (the
    # two sizes around it), cut rows of 1 KB never.
    import librett_amd as L
    copies = [c["desc"] for c in L.host_candidates(dim, [0, 2, 1], elem) if c["method"] == L.TILED_COPY]
    assert copies and all(d.endswith(" stream") == streamed for d in copies)


@pytest.mark.parametrize("dim,perm,elem,streamed", [
    ([4096, 6592], [1, 0], 4, False), ([4096, 6656], [1, 0], 4, True), ([4096, 3296], [1, 0], 8, False),
    ([4096, 3328], [1, 0], 8, True), ([1024, 103, 256], [0, 2, 1], 4, False), ([1024, 104, 256], [0, 2, 1], 4, True),
    ([2312, 115, 157], [0, 2, 1], 8, False), ([2312, 115, 159], [0, 2, 1], 8, True),
])
def test_inputs_that_the_cache_half_holds_do_not_stream(dim, perm, elem, streamed):
    # Whole lines at 103 and 104 MiB; rows of whole half lines at 318 and 322.5.
    import librett_amd as L
    method = L.TILED_COPY if perm[0] == 0 else L.TILED
    plans = [c["desc"] for c in L.host_candidates(dim, perm, elem) if c["method"] == method]
    assert any(d.endswith(" stream") for d in plans) == streamed
