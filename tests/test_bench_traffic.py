"""The benchmark's measured traffic is the reading of the kernel it names."""
import json
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_traffic_is_the_reported_kernels(tmp_path, monkeypatch):
    import bench
    with open(os.path.join(ROOT, "profiles", "traffic_solve_xi_1025x257.json")) as f:
        d = json.load(f)
    assert d["kernel"].split(" ")[0] == bench.SOLVE_KERNEL
    assert bench.measured_traffic() == d["bytes_per_launch"]
    assert d["bytes_per_launch"] >= d["algorithmic_bytes_per_launch"]
    # the scaled counters are what the file says they add up to
    total = 1024 * (d["fetch_size_kib_per_dispatch"] * d["fetch_scale"] + d["write_size_kib_per_dispatch"] * d["write_scale"])
    assert abs(total - d["bytes_per_launch"]) < 1e-4 * total
    # another kernel's reading is not reported
    other = tmp_path / "t.json"
    other.write_text(json.dumps(dict(d, kernel="k_other<double> (xi lines)")))
    monkeypatch.setattr(bench, "TRAFFIC_FILE", str(other))
    assert bench.measured_traffic() is None
    monkeypatch.setattr(bench, "TRAFFIC_FILE", str(tmp_path / "absent.json"))
    assert bench.measured_traffic() is None
