"""bench.py's counter summary: it reads the rows of the kernel that served the
probe's solves, and a run reports the traffic of its own kernel or none."""
import csv
import json

import pytest

import bench


def _counters(d, counter, rows):
    d.mkdir()
    with open(d / "x_counter_collection.csv", "w", newline="") as f:
        w = csv.writer(f)
        w.writerow(["Dispatch_Id", "Kernel_Name", "Counter_Name", "Counter_Value"])
        for i, (name, kib) in enumerate(rows):
            w.writerow([i, name, counter, kib])


@pytest.mark.parametrize("exchanges,kernel,name", [
    (1, "k_pcg_one", "void silk::amd::k_pcg_one<2, 6>(PersistDev, float)"),
    (2, "k_pcg_persistent", "void silk::amd::k_pcg_persistent<1>(PersistDev, float)")])
def test_summary_follows_the_kernel(exchanges, kernel, name, tmp_path, monkeypatch):
    monkeypatch.setattr(bench, "PROFILES", str(tmp_path / "profiles"))
    copy = 256 << 20
    pcg = [(name, 100.0), (name, 300.0)]
    # Fetches are counted at half, writes in full.
    _counters(tmp_path / "fetch", "FETCH_SIZE", pcg + [("k_copy_unless", copy / 2048)] * 3)
    _counters(tmp_path / "write", "WRITE_SIZE", pcg + [("k_copy_unless", copy / 1024)] * 3)
    log = tmp_path / "probe.log"
    log.write_text(json.dumps({"probe": "pmc", "steps": 2, "pcg_iterations": 10,
                               "copy_bytes": copy, "copy_reps": 3, "vertices": 6561,
                               "pcg_exchanges": exchanges}) + "\n")
    assert bench.pmc_summary(str(tmp_path / "fetch"), str(tmp_path / "write"), str(log)) == 0
    tr = bench.traffic_summary(kernel, 6561)
    assert tr["kernel"] == kernel and tr["pcg_launches"] == 2
    assert tr["bytes_per_iteration"] == pytest.approx(400 * 1024 * (2 + 1) / 10)
    other = {"k_pcg_one": "k_pcg_persistent", "k_pcg_persistent": "k_pcg_one"}[kernel]
    assert bench.traffic_summary(other, 6561) is None
    assert bench.traffic_summary(kernel, 100) is None
    assert bench.classes({"pcg_exchanges": exchanges})[1] == kernel
