"""The profile summary and what bench.py takes from it, on made-up profiler output: a
kernel launched at two sizes (one array, and three arrays together) has the rate of
all its bytes over all its time, and a single array's traffic comes from the
launches of one array."""
import csv
import json

import pytest

import bench
from waveletpotentials_amd import rocprof_summary as R

LP = ("void whhd::lp::lp_kernel<whhd::Wavelet<whhd::Ix{a}, whhd::UpCdf37, 0, 0, 4>, whhd::Wavelet<whhd::Ix{b}, "
      "whhd::UpCdf46, 0, 0, 5>, 8, false, 2>(whhd::lp::LpJobs)").format(a="HalfN", b="WholeD44")
CAL = "void at::vectorized_elementwise_kernel<4, MulFunctor<float>>(int)"
ONE, MERGED = 65792, 198144          # work-items
LAUNCHES = [ONE, ONE, ONE, MERGED]
US = {ONE: 30.0, MERGED: 72.0}
BYTES = {ONE: 68e6, MERGED: 210e6}   # either way


@pytest.fixture
def dirs(tmp_path):
    trace, fetch, write = (tmp_path / d for d in ("trace", "fetch", "write"))
    for d in (trace, fetch, write):
        d.mkdir()
    rows = [(LP, g) for g in LAUNCHES]

    def dump(path, head, lines):
        with open(path, "w", newline="") as f:
            w = csv.writer(f)
            w.writerow(head)
            w.writerows(lines)

    dump(trace / "run_kernel_stats.csv", ["Name", "Calls", "TotalDurationNs"],
         [[LP, len(rows), sum(US[g] for g in LAUNCHES) * 1e3], [CAL, 1, 5e4]])
    dump(trace / "run_kernel_trace.csv",
         ["Kernel_Name", "Grid_Size_X", "Grid_Size_Y", "Grid_Size_Z", "Start_Timestamp", "End_Timestamp"],
         [[n, g, 1, 1, 0, int(US[g] * 1e3)] for n, g in rows])
    for d in (fetch, write):
        dump(d / "run_counter_collection.csv", ["Kernel_Name", "Grid_Size", "Counter_Value"],
             [[n, g, BYTES[g] / 1024] for n, g in rows] + [[CAL, 1, R.CAL_BYTES / 1024]])
    return trace, fetch, write


def test_rate_of_a_kernel_with_two_launch_sizes(dirs):
    kernels, _, _, by_size = R.summarize(*map(str, dirs))
    (row,) = [v for k, v in kernels.items() if k.startswith("lp_kernel")]
    assert row["calls"] == 4
    rate = (row["fetch_bytes"] + row["write_bytes"]) / row["avg_us"]
    assert rate == pytest.approx(2 * sum(BYTES[g] for g in LAUNCHES) / sum(US[g] for g in LAUNCHES))
    assert {r["grid"]: r["fetch_bytes"] / r["avg_us"] for r in by_size} == pytest.approx(
        {g: BYTES[g] / US[g] for g in US})


def test_bench_takes_the_single_array_launch(dirs, tmp_path, monkeypatch):
    (tmp_path / "profiles").mkdir()
    R.write_outputs(*R.summarize(*map(str, dirs))[:3], str(tmp_path / "profiles" / "traffic_recover3d_256"), "cmd",
                    R.summarize(*map(str, dirs))[3])
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    algorithmic = 2 * 4 * 257 * ONE   # the pass of one array, lines of 257 samples
    got = bench.measured_traffic("lp_kernel<cdf4.6 d,L=8,inv,strided>", algorithmic)
    assert got["bytes"] == 2 * BYTES[ONE]
    assert bench.measured_traffic("lp_kernel<cdf4.6 d,L=8,fwd,strided>", algorithmic) is None
    with open(tmp_path / "profiles" / "traffic_recover3d_256.json") as f:
        assert {r["grid"] for r in json.load(f)["by_size"]} == {ONE, MERGED}
