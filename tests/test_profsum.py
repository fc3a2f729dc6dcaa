"""The profile summaries' rows: sweeps of all directions and of one, updates
after FP64 and FP32 sweeps, and the bench's lookup of a kernel's traffic."""
import csv
import os
import sys

import pytest

from festgpu import cases as C
from festgpu import profsum
from festgpu import roofline as R

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run(tmp_path, counter):
    """A counter CSV of two joint residuals of blocks of different sizes and
    one taken direction by direction between them, in FP64 and then in FP32;
    values 1, 2, ... per dispatch."""
    seq = []
    for t in ("double", "float"):
        k = f"void fest::k_sweeps<7, 3, false, {t}>(fest::Blk, fest::Sweeps, int, int)"
        u = "void fest::k_update<7>(fest::Blk, double, double, int)"
        seq += [(k, 3100), (u, 500), (k, 1000), (k, 1010), (k, 1090), (u, 500), (k, 900), (u, 300)]
    seq = [("fest::k_step_begin(fest::Blk, int)", 100)] + seq
    os.makedirs(tmp_path, exist_ok=True)
    with open(os.path.join(tmp_path, "x_counter_collection.csv"), "w", newline="") as f:
        w = csv.writer(f)
        w.writerow(["Dispatch_Id", "Grid_Size", "Kernel_Name", "Counter_Name", "Counter_Value"])
        for n, (name, grid) in enumerate(seq):
            w.writerow([n + 1, grid, name, counter, n + 1.0])
    return len(seq)


def test_launches_apart(tmp_path):
    run(tmp_path, "FETCH_SIZE")
    got = profsum.counters(str(tmp_path), "FETCH_SIZE")
    name = "k_sweeps<7, 3, false, %s> %s"
    want = {("step_begin", "k_step_begin"): 1.0, ("update", "k_update<7>"): 19.0 / 3,
            ("update", "k_update<7> after float sweeps"): 43.0 / 3}
    for t, first in (("double", 2), ("float", 10)):
        want["flux", name % (t, "all directions")] = first + 3.0
        for d, v in zip("ijk", (2, 3, 4)):
            want["flux_" + d, name % (t, d)] = float(first + v)
    assert got == pytest.approx(want)


def test_only_single_directions():
    rows = [(n, "k_update<5>" if n % 4 == 0 else "k_sweeps<5, 1, false, double>") for n in range(12)]
    got = profsum.launches(rows)
    assert [got[n][0] for n in range(12)] == ["update", "flux_i", "flux_j", "flux_k"] * 3


def test_traffic_rows(tmp_path):
    run(tmp_path / "f", "FETCH_SIZE")
    run(tmp_path / "w", "WRITE_SIZE")
    text = profsum.traffic(str(tmp_path / "f"), str(tmp_path / "w"), "sst_bump_16x12x8")
    rows = [[c.strip() for c in line.strip("|").split("|")] for line in text.splitlines() if line.startswith("| flux")]
    assert {r[0] for r in rows} == {"flux", "flux_i", "flux_j", "flux_k"}
    case = C.sst_bump(16, 12, 8)[0]
    joint = R.bytes_per_launch(case, "flux")
    assert max(R.bytes_per_launch(case, "flux_" + d) for d in "ijk") < joint
    assert joint < sum(R.bytes_per_launch(case, "flux_" + d) for d in "ijk")
    assert sum(len(r) == 4 and r[0] == "flux" and float(r[2]) == pytest.approx(joint, rel=1e-5) for r in rows) == 2


@pytest.mark.parametrize("group", ["flux_i", "flux_j", "flux_k", "grad", "update"])
def test_bench_finds_the_measured_traffic(group, monkeypatch):
    monkeypatch.setattr(sys, "argv", ["bench.py"])
    sys.path.insert(0, ROOT)
    import bench
    case = C.sst_bump(4, 4, 4)[0]
    case.name = "sst_bump_256x128x128"
    case.imx, case.jmx, case.kmx = 257, 129, 129
    got = bench.measured_traffic(case, group)
    assert got is not None
    # between the bytes without which it cannot do, halved by the last-level cache, and twice them
    assert 0.5 < got / R.bytes_per_launch(case, group) < 2.0
