"""bench.py's traffic figures: profiles/traffic.json against the kernels the workloads name. No GPU."""
import importlib.util
import json
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
spec = importlib.util.spec_from_file_location("bench_under_test", os.path.join(ROOT, "bench.py"))
bench = importlib.util.module_from_spec(spec)
spec.loader.exec_module(bench)
with open(os.path.join(ROOT, "profiles", "traffic.json")) as f:
    TRAFFIC = json.load(f)["traffic"]


@pytest.mark.parametrize("name", sorted(TRAFFIC))
def test_traffic_is_of_the_kernels_that_run(name):
    wl = bench.make_workloads()[name]
    assert bench.measured_traffic(wl) == sum(TRAFFIC[name].values())


def test_traffic_of_another_kernel_is_not_printed():
    wl = bench.make_workloads()["softmax_f16_8192x50257"]
    wl.kernel = "row_kernel"
    assert bench.measured_traffic(wl) is None
    wl.kernel = "softmax_long_kernel + another_kernel"
    assert bench.measured_traffic(wl) is None
    wl.name = "no such workload"
    assert bench.measured_traffic(wl) is None
