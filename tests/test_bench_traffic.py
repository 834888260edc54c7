"""The counter traffic that a benchmark line carries belongs to the launches it timed: a
launch configuration without a record names no kernel."""
import json
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402

PROFILES = os.path.join(bench.ROOT, "profiles")
RECORDS = [f[len("traffic_"):-len(".json")].rsplit("_", 1) for f in sorted(os.listdir(PROFILES))
           if f.startswith("traffic_") and f.endswith(".json")]


@pytest.mark.parametrize("workload,solver", RECORDS, ids=lambda p: p)
def test_traffic_names_the_kernel_that_was_counted(workload, solver):
    with open(os.path.join(PROFILES, f"traffic_{workload}_{solver}.json")) as f:
        record = json.load(f)
    for entry in record["by_launch_config"]:
        bytes_, kernel, note = bench.traffic_for(workload, solver, entry["launch_config"])
        assert (bytes_, kernel, note) == (entry["bytes_per_iteration"], record["kernel"], None)
    bytes_, kernel, note = bench.traffic_for(workload, solver, ["no such launch", 0, True])
    assert bytes_ is None and kernel is None and "no such launch" in note
