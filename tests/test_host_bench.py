"""The HBM traffic that bench.py prints belongs to the kernel it times (CPU
only): profiles/traffic.json names the kernel, with the bytes of that kernel's
row in the profile, and another kernel has none."""
import os
import re
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


def test_traffic_is_the_timed_kernels():
    got = bench.load_traffic(bench.PHYS_KERNEL)
    with open(os.path.join(ROOT, "profiles", "traffic_timestep_L170_N96.md")) as f:
        rows = [line.split("|") for line in f if line.startswith("| `")]
    row = [r for r in rows if re.match(r" `%s\b" % bench.PHYS_KERNEL, r[1])]
    assert len(row) == 1
    assert abs(got / 1e6 - float(row[0][5])) <= 0.06
    assert bench.load_traffic("phys") is None
