"""What bench.py reports of a run: the kernel it names is the one the configuration that ran has, and
the bytes of its roofline are no more than the kernels were measured to move. (On the CPU.)"""
import importlib.util
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location("bench_under_test", os.path.join(ROOT, "bench.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


@pytest.mark.parametrize("runs,two,f32,name", [
    ((1, 64, 8), 1, False, "k_step_lane64<0, 8>"), ((1, 64, 8), 2, False, "k_step2_lane64<0, 8>"),
    ((4, 64, 1), 1, False, "k_step<0, false, double, 64>"), ((4, 128, 4), 1, False, "k_step_refill<0, double, 128, 4>"),
    ((1, 64, 4), 1, True, "k_step_lane<0, 64, 4>"), ((1, 64, 4), 2, True, "k_step_lane2<0, 64, 4>"),
    ((4, 256, 1), 1, True, "k_step<0, false, float, 256>")])
def test_kernel_names(bench, runs, two, f32, name):
    tune = {"lanes_per_cru": runs[0], "block": runs[1], "crus_per_lane": runs[2], "steps_per_launch": two}
    assert bench.kernel_name(tune, f32) == name


@pytest.mark.parametrize("form", ["fp64", "fp64_pair", "fp32", "fp32_pair"])
def test_roofline_bytes_are_moved(bench, form):
    counted = bench.STATE_BYTES_F32 if form.startswith("fp32") else bench.STATE_BYTES
    moved = bench.measured_traffic(1000, form) / 1000
    assert 0.9 * moved < counted <= moved
    assert 0.0 < bench.profile_value("valu_busy", form) < 1.0
