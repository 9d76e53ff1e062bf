"""The rule that chooses the running launch configuration (gw_route.h) on a whole
device and on a part of it: every crossing lies in proportion to the compute
units, and everything else is as on the whole. (On the CPU.)"""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "gw_route.h"
#include <cstdio>
int main()
{
    int cfg, f32, cells, cus;
    long long crus;
    while (std::scanf("%d %d %lld %d %d", &cfg, &f32, &crus, &cells, &cus) == 5) {
        const gw::BatchSize b{f32 != 0, crus, cells, cus};
        const int r = gw::route(cfg, b);
        const gw::LaunchCfg &L = gw::kConfigs[r];
        std::printf("%d %d %d %d\n", L.lanes, L.threads, L.cpl, gw::route_pair(r, b) ? 2 : 1);
    }
}
"""
CONFIGS = [(4, 64, 1), (4, 128, 1), (4, 256, 1), (4, 512, 1)] + [(1, t, c) for c in (1, 2, 4, 8) for t in (64, 128, 256)] + \
          [(4, 64, 2), (4, 64, 4), (4, 128, 4), (4, 256, 4)]


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    d = tmp_path_factory.mktemp("route")
    (d / "route.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{os.path.join(ROOT, 'gw-model_amd', 'csrc')}",
                    str(d / "route.cpp"), "-o", str(d / "route")], check=True)

    def run(rows):
        """[(shape, FP32-local, CRUs, cells, compute units)] -> [(running shape, steps per launch)]"""
        text = "".join(f"{CONFIGS.index(s)} {int(f)} {n} {c} {u}\n" for s, f, n, c, u in rows)
        out = subprocess.run([str(d / "route")], input=text, capture_output=True, text=True, check=True).stdout
        return [(tuple(int(x) for x in ln.split()[:3]), int(ln.split()[3])) for ln in out.splitlines()]

    return run


# (shape asked for, FP32-local, CRUs and cells of 256 compute units at the crossing, what runs below it and from it on)
CROSSINGS = [
    ((4, 512, 1), False, 180_000, 1, (4, 256, 1), (4, 64, 1)),
    ((4, 64, 1), False, 340_000, 1, (4, 64, 1), (1, 64, 2)),
    ((4, 64, 4), False, 340_000, 1, (4, 64, 4), (1, 64, 2)),
    ((4, 256, 1), False, 950_000, 64, (1, 64, 2), (1, 64, 4)),
    ((4, 256, 1), False, 2_500_000, 64, (1, 64, 4), (1, 64, 8)),
    ((4, 128, 1), True, 350_000, 1, (4, 256, 1), (4, 64, 1)),
    ((1, 64, 4), True, 300_000, 1, (1, 64, 1), (1, 64, 4)),
    ((1, 256, 8), True, 300_000, 1, (1, 256, 1), (1, 256, 8)),
]


@pytest.mark.parametrize("cus", [256, 128, 64, 32])
def test_crossings_lie_in_proportion_to_the_compute_units(route, cus):
    for shape, f32, crus, cells, below, above in CROSSINGS:
        at = crus * cus // 256
        (a, _), (b, _) = route([(shape, f32, at - 1, cells, cus), (shape, f32, at, cells, cus)])
        assert (a, b) == (below, above), (shape, f32, at)
    many = 256 * cus // 256   # cells
    assert [r for r, _ in route([((4, 256, 1), False, 10 * many, many - 1, cus), ((4, 256, 1), False, 10 * many, many, cus)])] == \
        [(4, 256, 1), (4, 64, 1)]
    two = 450_000 * cus // 256
    assert [s for _, s in route([((1, 64, 4), True, two - 1, 1, cus), ((1, 64, 4), True, two, 1, cus)])] == [1, 2]
    # FP64 lanes only where cells fill a wave on average, on any device
    n = 340_000 * cus // 256
    assert [r for r, _ in route([((4, 256, 1), False, n, n // 64, cus), ((4, 256, 1), False, n, n // 64 + 1, cus)])] == \
        [(1, 64, 2), (4, 64, 1)]


def test_shapes_that_run_as_themselves(route):
    one = [s for s in CONFIGS if s[0] == 1 and s[2] == 1]
    assert [r for r, _ in route([(s, True, n, 1, 256) for s in one for n in (1, 1_000_000)])] == [s for s in one for _ in (0, 1)]
    refilled = [s for s in CONFIGS if s[0] == 1 and s[2] > 1]
    assert [r for r, _ in route([(s, True, 1_000_000, 1, 256) for s in refilled])] == refilled
    assert [r for r, _ in route([(s, True, 1000, 1, 256) for s in refilled])] == [(1, t, 1) for _, t, _ in refilled]
