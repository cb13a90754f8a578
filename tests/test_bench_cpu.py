"""Host logic of bench.py that needs no GPU: the one-GPU rule and the
profile summaries that `roofline.traffic` and the kernel-time tables come
from (rocprofv3 CSV in, scaled bytes and tables out)."""
import csv
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


def test_more_than_one_gpu_is_refused_with_a_message():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 2
    assert "single MI355X" in r.stderr and r.stdout == ""


def _write_pmc(d, rows):
    os.makedirs(d, exist_ok=True)
    with open(os.path.join(d, "x_counter_collection.csv"), "w", newline="") as f:
        w = csv.DictWriter(f, fieldnames=["Dispatch_Id", "Kernel_Name", "Counter_Name", "Counter_Value",
                                          "Start_Timestamp", "End_Timestamp"])
        w.writeheader()
        for k, (name, counter, value, ns) in enumerate(rows):
            w.writerow({"Dispatch_Id": k, "Kernel_Name": name, "Counter_Name": counter, "Counter_Value": value,
                        "Start_Timestamp": 1000, "End_Timestamp": 1000 + ns})


def test_traffic_summary_counts_requests_by_size(tmp_path):
    """Reads are the requests of each size times that size -- a streaming
    copy's 128-byte requests and a gather's 64-byte ones alike, with no factor
    of one applied to the other; WRITE_SIZE is KiB per dispatch."""
    copy = 1 << 30
    trace = "void dl::k_trace_queue<false>(dl::BvhView, dl::RenderBufs, int*)"
    rows = []
    for name, per_dispatch in ((trace, [(10, 300, 40), (30, 100, 80)]), ("k_copy", [(0, 0, copy // 128)])):
        for ns, r in zip((2_000_000, 4_000_000), per_dispatch):
            rows += [(name, "TCC_EA0_RDREQ_%dB_sum" % b, v, ns) for b, v in zip((32, 64, 128), r)]
    _write_pmc(str(tmp_path / "f"), rows)
    _write_pmc(str(tmp_path / "w"), [(trace, "WRITE_SIZE", 2.0, 1), ("k_copy", "WRITE_SIZE", copy / 1024.0, 1)])
    out = tmp_path / "traffic.json"
    bench.summarize_pmc(str(tmp_path / "f"), str(tmp_path / "w"), str(out), copy_bytes=copy, commands="cmd")
    t = json.loads(out.read_text())
    assert t["copy_fetch"] == 1.0 and t["copy_write"] == 1.0
    k = t["kernels"]["k_trace_queue<false>"]
    assert k["launches"] == 2 and k["ms"] == pytest.approx(3.0)
    assert k["fetch_bytes"] == 20 * 32 + 200 * 64 + 60 * 128 and k["write_bytes"] == 2048
    assert k["gbs"] == pytest.approx((k["fetch_bytes"] + 2048) / 3e-3 / 1e9)


def test_roofline_fraction_is_of_measured_traffic():
    """The fraction of the HBM peak comes from the profiled launches' traffic;
    bytes that caches may have served (here 9 TB/s of them) are only listed."""
    r = bench.roofline("k_x", "closest hit", 4e9, 1.0, 9e9, 1000.0, 8.0, 3.0, 1000.0, 10, False)
    assert r["achieved"] == 4000.0 and r["frac"] == 0.5
    assert r["queries"]["touched_gbs"] == 9000.0 and r["queries"]["launches"] == 10
    r = bench.roofline("k_x", "closest hit", None, None, 9e9, 1000.0, 8.0, 3.0, 1000.0, 10, False)
    assert r["achieved"] is None and r["frac"] is None


def test_kernel_time_table(tmp_path):
    d = tmp_path / "prof"
    d.mkdir()
    with open(d / "bench_kernel_stats.csv", "w", newline="") as f:
        w = csv.DictWriter(f, fieldnames=["Name", "Calls", "TotalDurationNs", "AverageNs", "MinNs", "MaxNs",
                                          "Percentage"])
        w.writeheader()
        w.writerow({"Name": "void dl::k_trace_queue<false>(dl::BvhView, dl::RenderBufs, int*)", "Calls": 4,
                    "TotalDurationNs": 8e6, "AverageNs": 2e6, "MinNs": 1e6, "MaxNs": 3e6, "Percentage": 80.0})
    out = tmp_path / "stats.md"
    bench.summarize_stats(str(d), str(out), "cmd", "title")
    text = out.read_text()
    assert "# Kernel time: title" in text and "```\ncmd\n```" in text
    assert "| k_trace_queue<false> | 4 | 8.00 | 2000.0 | 1000.0 | 3000.0 | 80.00 |" in text
