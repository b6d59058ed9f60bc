"""The traffic table of the ray-query kernel counts a query's launches together."""
import csv

import pytest

import bench

COPY = "__amd_rocclr_copyBuffer"
NS = "void rtgpu::(anonymous namespace)::"
FIRST = NS + "k_trace_persistent<44, 16, false, false, false, false, false>(rtgpu::(anonymous namespace)::TraceArgs)"
MARKED = NS + "k_trace_persistent<4, 16, false, false, false, false, true>(rtgpu::(anonymous namespace)::TraceArgs)"
TEAMS = NS + "k_trace_marked<false>(rtgpu::(anonymous namespace)::TraceArgs)"
DIRECT = NS + "k_trace_direct<44, 4, false, false>(rtgpu::(anonymous namespace)::TraceArgs)"
ZERO = NS + "k_zero_counter(unsigned int*)"


def _write(path, counter, rows):
    with open(path, "w", newline="") as f:
        w = csv.DictWriter(f, ["Dispatch_Id", "Counter_Name", "Kernel_Name", "Counter_Value"])
        w.writeheader()
        for i, (k, v) in enumerate(rows):
            w.writerow({"Dispatch_Id": i, "Counter_Name": counter, "Kernel_Name": k, "Counter_Value": v})


def test_a_marked_launch_counts_with_its_query(tmp_path):
    copies = [(COPY, float(1 << 19))] * 5  # half of the copied KiB: a scale of 2
    queries = [(DIRECT, 100.0), (ZERO, 1.0), (FIRST, 40.0), (MARKED, 2.0), (ZERO, 1.0), (FIRST, 50.0), (TEAMS, 3.0)]
    _write(tmp_path / "f.csv", "FETCH_SIZE", copies + queries)
    _write(tmp_path / "w.csv", "WRITE_SIZE", [(COPY, float(1 << 20))] * 5 + queries)
    t = bench.traffic_table(tmp_path / "f.csv", tmp_path / "w.csv", ["a", "b", "c"], "", out=tmp_path / "t.json")
    got = {c: (e["kernel"], e["traffic_bytes"]) for c, e in t["configs"].items()}
    assert got == {"a": (DIRECT, 300 * 1024), "b": (FIRST, 126 * 1024), "c": (FIRST, 159 * 1024)}


def test_a_launch_too_few_is_refused(tmp_path):
    rows = [(COPY, 1.0)] * 5 + [(FIRST, 1.0), (MARKED, 1.0)]
    _write(tmp_path / "f.csv", "FETCH_SIZE", rows)
    _write(tmp_path / "w.csv", "WRITE_SIZE", rows)
    with pytest.raises(AssertionError):
        bench.traffic_table(tmp_path / "f.csv", tmp_path / "w.csv", ["a", "b"], "", out=tmp_path / "t.json")
