"""The recorded HBM traffic that the benchmark publishes beside its rooflines (profiles/traffic.json): no
kernel group can move less than the intermediates it writes and reads.  T is written once by the
GEMM stages and read by the term sum, S the other way round."""
import json
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("workload", ["qc", "qc3"])
def test_recorded_traffic_covers_the_intermediates(workload):
    records = json.load(open(os.path.join(ROOT, "profiles", "traffic.json")))[workload]
    assert len(records) == 2
    for name, r in records.items():
        t, s = 8e-9 * r["t_elements"], 8e-9 * r["s_elements"]
        written, read = (t, s) if name.startswith("gemm") else (s, t)
        assert r["write_gb"] >= written and r["fetch_gb"] >= read, name
