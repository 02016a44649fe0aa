"""bench.py's VALU figures (no GPU): shares of what the VALU can issue, never
above one."""
import csv
import json
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)


def test_issue_fraction_of_the_fastest_measured_rate(tmp_path):
    """Multiply-adds from eight waves issue 0.45 a cycle and SIMD, half lanes
    here: a share of 0.9 of one every two cycles."""
    k = "void vz::(anonymous namespace)::k_path<false, (vz::(anonymous namespace)::PathSrc)0>(vz::PathGroup)"
    cycles = 1e6
    insts = 0.45 * cycles * 1024
    vals = {"SQ_INSTS_VALU": insts, "SQ_ACTIVE_INST_VALU": insts, "SQ_THREAD_CYCLES_VALU": 32 * insts,
            "SQ_BUSY_CYCLES": 32 * cycles}
    with open(tmp_path / "sq.csv", "w", newline="") as f:
        w = csv.writer(f, quoting=csv.QUOTE_NONNUMERIC)
        w.writerow(["Kernel_Name", "Counter_Name", "Counter_Value"])
        for name, v in vals.items():
            w.writerow([k, name, v])
    js = tmp_path / "sq.json"
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--summarize-sq", str(tmp_path / "sq.csv"),
                        "--sq-map", "k_path<false, (vz::(anonymous namespace)::PathSrc)0>=book", "--out-md",
                        str(tmp_path / "sq.md"), "--out-json", str(js), "--commands", "cmd"], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    e = json.load(open(js))["book"]
    assert e["valu_issue_frac"] == 0.9 and e["lanes_active"] == 0.5
    import bench
    ms = cycles / 2.4e9 * 1e3
    roof = bench.valu_roofline(e, ms)
    assert abs(roof["frac"] - 0.45) < 1e-3  # half the lanes of 0.9


def test_committed_profiles_hold_shares():
    for e in json.load(open(os.path.join(ROOT, "profiles", "path_kernel_sq.json"))).values():
        assert 0.0 < e["valu_issue_frac"] <= 1.0 and 0.0 < e["lanes_active"] <= 1.0
