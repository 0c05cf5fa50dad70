"""bench.py's traffic summary of profiler counters: every kernel that runs a
plan is a case of its own, whatever its tile form."""
import csv
import json

import pytest

import bench

KERNELS = ["lrt::k_tiled<4, 128, 128, 4, 4, false, true>", "lrt::k_copy<4, 1, true>", "lrt::k_narrow<lrt::NarrowOps<4, 256, 8>, true>",
           "lrt::k_skew<8, 32, 64, 256, true, true>", "lrt::k_copy<8, 2, true>", "lrt::k_packed<8, 2>",
           "lrt::k_tiled<8, 64, 64, 2, 2, false, true>"]


def run_dir(path, factor, kernels):
    """A counter run that counted 1 / factor of each dispatch's KiB."""
    path.mkdir()
    n = [bench.np.prod(d) * float(e) for d, _, e in bench.CASES]
    rows = [("void %s(args)" % k, 256, b) for k, b in zip(kernels, n)] + [("void lrt::k_devcopy<1, true>(args)", 1 << 20, 16.0 * (1 << 20))]
    with open(path / "run_counter_collection.csv", "w", newline="") as fh:
        w = csv.writer(fh)
        w.writerow(["Dispatch_Id", "Kernel_Name", "Grid_Size", "Counter_Name", "Counter_Value"])
        for i, (k, g, b) in enumerate(rows):
            w.writerow([i, k, g, "C", b / 1024 / factor])
    return str(path)


def test_every_plan_kernel_is_a_case(tmp_path, capsys):
    log = tmp_path / "log"
    log.write_text("".join("plan (x) -> plan%d (1.0 ms)\n" % i for i in range(7)))
    f, w = run_dir(tmp_path / "f", 2.0, KERNELS), run_dir(tmp_path / "w", 1.0, KERNELS)
    bench.pmc_summary(f, w, str(log), str(tmp_path / "out.json"))
    got = json.load(open(tmp_path / "out.json"))["cases"]
    assert [c["kernel"] for c in got] == ["void %s(args)" % k for k in KERNELS]
    assert [c["plan"] for c in got] == ["plan%d" % i for i in range(7)]
    assert all(c["ratio"] == c["read_ratio"] == c["write_ratio"] == 1.0 for c in got)


def test_a_missing_case_is_an_error(tmp_path):
    f, w = run_dir(tmp_path / "f", 2.0, KERNELS[:6]), run_dir(tmp_path / "w", 1.0, KERNELS[:6])
    with pytest.raises(SystemExit):
        bench.pmc_summary(f, w, "/dev/null")
