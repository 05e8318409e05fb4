"""The counter-traffic record of the planned launches: found for their
configuration only, the scaled counters, and named in the profile summary."""
import os

import pytest

import bench

PLANNED = {"kernel": 2, "cols_per_thread": 2, "strip": 64, "segment": 171, "prefetch_rows": 1, "steps_per_launch": 7,
           "col_block": 2}


def test_planned_traffic_record():
    kv = dict(line.strip().split(": ", 1) for line in open(bench.TRAFFIC_FILES[1]))
    fetch, write = float(kv["fetch_size_kib_avg"]), float(kv["write_size_kib_avg"])
    traffic = float(kv["traffic_bytes_per_launch"])
    assert traffic == pytest.approx((float(kv["fetch_scale"]) * fetch + float(kv["write_scale"]) * write) * 1024, rel=1e-6)
    assert bench.measured_traffic(PLANNED) == traffic
    for key, other in (("segment", 128), ("steps_per_launch", 6), ("col_block", 8)):
        assert bench.measured_traffic({**PLANNED, key: other}) != traffic
    md = open(os.path.join(bench.ROOT, "profiles", "fom_fusedW_config2_fp64.md")).read()
    assert kv["kernel"] in md and f"{fetch:,.1f}" in md and f"{write:,.1f}" in md
