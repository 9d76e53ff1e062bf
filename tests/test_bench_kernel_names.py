"""The kernel that bench.py names is the one the configuration that ran has. (On the CPU.)"""
import importlib.util
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("runs,two,f32,name", [
    ((1, 64, 8), 1, False, "k_step_lane64<0, 8>"), ((1, 64, 8), 2, False, "k_step2_lane64<0, 8>"),
    ((4, 64, 1), 1, False, "k_step<0, false, double, 64>"), ((4, 128, 4), 1, False, "k_step_refill<0, double, 128, 4>"),
    ((1, 64, 4), 1, True, "k_step_lane<0, 64, 4>"), ((1, 64, 4), 2, True, "k_step_lane2<0, 64, 4>"),
    ((4, 256, 1), 1, True, "k_step<0, false, float, 256>")])
def test_kernel_names(runs, two, f32, name):
    spec = importlib.util.spec_from_file_location("bench_under_test", os.path.join(ROOT, "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    tune = {"lanes_per_cru": runs[0], "block": runs[1], "crus_per_lane": runs[2], "steps_per_launch": two}
    assert bench.kernel_name(tune, f32) == name
