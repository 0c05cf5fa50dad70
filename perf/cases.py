"""The work that users of this library have it do, as cases that a timing harness can run.

Three kinds of case, each through the package's public entry points:

  single  one plan, executed again and again: librettPlan + librettExecute;
          with "back" a second plan takes the result back to the input's
          order, as a program does around a contraction or an FFT
  batch   many independent transposes in one launch: Batch(...).execute()
  serve   a burst of requests to the serving engine: Server.submit / wait

Tensors are column-major in the library's sense (dim[0] varies fastest), so a
torch tensor of them has the dims reversed. Elements are float32, float64 or
complex128 (4, 8 or 16 bytes), uniform in [-1, 1).

One pass moves every element once and computes nothing, so work() counts each
input byte read once and each output byte written once, and no flops.
"""
import math
import os

import numpy as np
import torch

import librett_amd as L
from librett_amd import workloads

ELEMS = {4: torch.float32, 8: torch.float64, 16: torch.complex128}
# Each problem of a batch or burst starts on a 256-byte boundary of one big
# buffer, as allocations do.
ALIGN = 256
# The largest single transposes (and the largest request of a burst), bytes
# of the input: the size of the named benchmark problems.
SINGLE_MAX = 256 << 20
# Elements of one batched problem: the batched workload's range.
BATCH_VOL = (1e3, 1e6)
# Bytes of one served request: the serving workload's range.
SERVE_BYTES = (4 << 10, 64 << 20)


# Small tensors are timed there and back: one launch of a few microseconds
# alone says little.
BACK_BELOW = 8 << 20


def single(name, dim, perm, elem):
    return {"name": name, "kind": "single", "dim": ",".join(map(str, dim)), "perm": ",".join(map(str, perm)),
            "elem": elem, "back": math.prod(dim) * elem < BACK_BELOW}


def listed():
    return [
        # The smallest calls: a tensor of the size of the smoke test, there and back. Launch and latency are all
        # there is.
        single("tiny f64 rank 3", [64, 48, 32], [2, 0, 1], 8),
        # A few megabytes with odd dims, as in an application's inner loop (every dim odd, so no wide lanes).
        single("small f32 odd rank 4", [37, 51, 29, 21], [3, 1, 0, 2], 4),
        # Double-complex tensors of quantum chemistry, some 50 MB.
        single("mid c128 rank 4", [48, 36, 40, 45], [2, 0, 3, 1], 16),
        # The square matrix of the headline benchmark: 256 MiB, both dims line-aligned.
        single("matrix f32", [8192, 8192], [1, 0], 4),
        # Six powers of two, dims scattered: short leading dims on both sides.
        single("scatter f32 rank 6", [2, 8, 16, 32, 64, 128], [5, 3, 1, 0, 2, 4], 4),
        # The first dim stays first: rows move whole.
        single("rows f32", [1024, 256, 256], [0, 2, 1], 4),
        # The same with rows of an odd length, which end inside cache lines.
        single("rows odd f64", [2307, 115, 126], [0, 2, 1], 8),
        # Ragged rank 4 of the headline benchmark: a short first dim, odd runs on both sides.
        single("ragged f64 rank 4", [5, 97, 211, 331], [3, 1, 0, 2], 8),
        # Reversal of a rank-5 tensor of the transpose literature (TTC suite), 800 MB of traffic.
        single("reverse f64 rank 5", [48, 28, 28, 28, 48], [4, 3, 2, 1, 0], 8),
        # A short odd first dim that moves to the back (array of structures to structure of arrays).
        single("short dim f32", [7, 1483, 6465], [1, 2, 0], 4),
        # The batched workload: 4096 problems of rank 3-5, 1e3-1e6 elements, f64 and c128, in one launch.
        {"name": "batch 4096", "kind": "batch", "count": 4096, "seed": 20261202},
        # A burst of requests to the serving engine, 4 KiB to 64 MiB, rank 2-6, all element sizes.
        {"name": "serve burst 128", "kind": "serve", "count": 128, "seed": 7},
    ]


def draw(rng):
    """One more case: sizes spread over the logarithm of the whole range."""
    u = rng.random()
    seed = rng.randrange(1 << 30)
    if u < 0.12:
        return {"kind": "batch", "count": int(round(math.exp(rng.uniform(math.log(32), math.log(3600))))),
                "seed": seed}
    if u < 0.22:
        return {"kind": "serve", "count": rng.randrange(16, 129), "seed": seed}
    elem = rng.choice((4, 4, 8, 8, 16))
    nbytes = math.exp(rng.uniform(math.log(64 << 10), math.log(SINGLE_MAX)))
    if rng.random() < 0.5:
        # The three shapes of the large benchmark problems, at any size from 4 MiB.
        nbytes = max(nbytes, 4 << 20)
        dim, perm = workloads.large_case(seed, elem, rng.choice(("keep", "move", "small")), int(nbytes))
    else:
        vol = nbytes / elem
        dim, perm, _ = workloads.random_problem(np.random.default_rng(seed), 2, 6, vol, vol, [elem])
    while math.prod(dim) * elem > 1.02 * SINGLE_MAX:
        k = dim.index(max(dim))
        dim[k] = max(2, dim[k] * 7 // 8)
    c = single("", dim, perm, elem)
    del c["name"]
    return c


def _problems(case):
    """(dims, perm, element bytes) of each problem of a batch or burst."""
    rng = np.random.default_rng(case["seed"])
    got = []
    for _ in range(case["count"]):
        if case["kind"] == "batch":
            got.append(workloads.random_problem(rng, 3, 5, *BATCH_VOL, [8, 16]))
        else:
            elem = int(rng.choice([4, 8, 16]))
            got.append(workloads.random_problem(rng, 2, 6, SERVE_BYTES[0] / elem, SERVE_BYTES[1] / elem, [elem]))
    return got


def _one(case):
    return [int(x) for x in case["dim"].split(",")], [int(x) for x in case["perm"].split(",")], case["elem"]


def _offsets(problems):
    """Byte offset of each problem in one buffer, and the buffer's size."""
    at, total = [], 0
    for dim, _, elem in problems:
        at.append(total)
        total += -(-math.prod(dim) * elem // ALIGN) * ALIGN
    return at, total


_PROCESS = {}


def _library():
    """The library, on torch's own HIP runtime: a process has one runtime, and streams and pointers belong to it."""
    if "lib" not in _PROCESS:
        before = os.environ.get("ROCM_PATH")
        os.environ["ROCM_PATH"] = os.path.dirname(torch.__file__)
        try:
            _PROCESS["lib"] = L.lib()
        finally:
            if before is None:
                del os.environ["ROCM_PATH"]
            else:
                os.environ["ROCM_PATH"] = before
        torch.cuda.init()
        _PROCESS["stream"] = torch.cuda.Stream()
        L.librettInitialize()
    return _PROCESS["stream"]


def _server():
    """One serving engine per process, as a service has."""
    _library()
    if "server" not in _PROCESS:
        _PROCESS["server"] = L.Server(1 << 30)
    return _PROCESS["server"]


def _uniform(n, dtype, seed):
    """n values in [-1, 1), on the GPU."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    if dtype == torch.complex128:
        return torch.view_as_complex(torch.rand(n, 2, generator=g, device="cuda", dtype=torch.float64).mul_(2).sub_(1))
    return torch.rand(n, generator=g, device="cuda", dtype=dtype).mul_(2).sub_(1)


class _Plan:
    """A stored plan, destroyed with its owner."""

    def __init__(self, dim, perm, elem, stream):
        r, self.handle = L.librettPlan(len(dim), dim, perm, elem, stream)
        if r != L.LIBRETT_SUCCESS:
            raise RuntimeError("librettPlan failed: %d" % r)

    def __del__(self):
        if getattr(self, "handle", None) is not None:
            L.librettDestroy(self.handle)


class _BatchPlan:
    """A planned batch with its buffers, destroyed with its owner."""

    def __init__(self, problems, stream, inputs, outputs):
        self.batch = L.Batch(problems, stream)
        self.batch.set_buffers(inputs, outputs)

    def __del__(self):
        if hasattr(self, "batch"):
            self.batch.destroy()


def prepare(case, seed):
    stream = _library()
    with torch.cuda.stream(stream):
        if case["kind"] == "single":
            dim, perm, elem = _one(case)
            x = _uniform(math.prod(dim), ELEMS[elem], seed).view(dim[::-1])
            y = torch.empty([dim[p] for p in perm[::-1]], dtype=ELEMS[elem], device="cuda")
            state = {"kind": "single", "x": x, "y": y, "plan": _Plan(dim, perm, elem, stream.cuda_stream)}
            if case["back"]:
                inverse = [perm.index(i) for i in range(len(dim))]
                state["z"] = torch.empty_like(x)
                state["inverse"] = _Plan([dim[p] for p in perm], inverse, elem, stream.cuda_stream)
        else:
            problems = _problems(case)
            at, total = _offsets(problems)
            x = _uniform(total // 4, torch.float32, seed) if case["kind"] == "serve" else \
                _uniform(total // 8, torch.float64, seed)
            y = torch.zeros_like(x)
            inputs, outputs = [x.data_ptr() + o for o in at], [y.data_ptr() + o for o in at]
            state = {"kind": case["kind"], "x": x, "y": y}
            if case["kind"] == "batch":
                state["plan"] = _BatchPlan(problems, stream.cuda_stream, inputs, outputs)
            else:
                state["server"] = _server()
                state["requests"] = [(d, p, e, i, o) for (d, p, e), i, o in zip(problems, inputs, outputs)]
    # The plan runs on `stream` and the server on streams of its own: inputs are ready before either starts.
    stream.synchronize()
    return state


def run(state):
    if state["kind"] == "single":
        r = L.librettExecute(state["plan"].handle, state["x"].data_ptr(), state["y"].data_ptr())
        if r != L.LIBRETT_SUCCESS:
            raise RuntimeError("librettExecute failed: %d" % r)
        if "z" in state:
            r = L.librettExecute(state["inverse"].handle, state["y"].data_ptr(), state["z"].data_ptr())
            if r != L.LIBRETT_SUCCESS:
                raise RuntimeError("librettExecute failed: %d" % r)
            return state["y"], state["z"]
    elif state["kind"] == "batch":
        r = state["plan"].batch.execute()
        if r != L.LIBRETT_SUCCESS:
            raise RuntimeError("batch execute failed: %d" % r)
    else:
        server = state["server"]
        tickets = [server.submit(*q) for q in state["requests"]]
        for t in tickets:
            server.wait(t)
    return state["y"]


def work(case):
    if case["kind"] == "single":
        dim, _, elem = _one(case)
        n = math.prod(dim) * elem * (2 if case["back"] else 1)
    else:
        n = sum(math.prod(d) * e for d, _, e in _problems(case))
    return {"bytes": 2 * n, "flops": 0}


def _permuted(x, dim, perm):
    """The library's permutation of a flat tensor, by torch."""
    r = len(dim)
    return x.view(dim[::-1]).permute([r - 1 - perm[r - 1 - t] for t in range(r)]).contiguous()


def exact(case, seed):
    """Every element in its new place: the values are copied, so 64 bits hold them exactly."""
    with torch.cuda.stream(_library()):
        if case["kind"] == "single":
            dim, perm, elem = _one(case)
            x = _uniform(math.prod(dim), ELEMS[elem], seed)
            y = _permuted(x, dim, perm)
            if elem == 4:
                x, y = x.double(), y.double()
            if case["back"]:
                y = (y, x.view(dim[::-1]))
        else:
            problems = _problems(case)
            at, total = _offsets(problems)
            x = _uniform(total // 4, torch.float32, seed) if case["kind"] == "serve" else \
                _uniform(total // 8, torch.float64, seed)
            y = torch.zeros_like(x)
            xb, yb = x.view(torch.uint8), y.view(torch.uint8)
            for (dim, perm, elem), o in zip(problems, at):
                n = math.prod(dim) * elem
                yb[o:o + n] = _permuted(xb[o:o + n].view(ELEMS[elem]), dim, perm).view(-1).view(torch.uint8)
            y = y.double() if case["kind"] == "serve" else y
    torch.cuda.synchronize()
    return y
