"""Kernels that only batches of some size run (gw_batch_get_running says which
ran): each in a batch large enough for it, against the same cells elsewhere."""
import numpy as np
import pytest

from .test_gpu_lane64 import SIZES, _cells, _open, _same, _state
from .test_gpu_parity import say

pytestmark = pytest.mark.gpu

KEYS = ("CaSS", "CaJSR", "LCC", "LCC_inactivation", "RyR", "ClCh", "JLCC")


def _pace(gwcapi):
    return {"kind": gwcapi.PROTO_PACE, "period": 500.0, "duration": 1.0, "amplitude": 100.0, "start": 0.0}


@pytest.mark.parametrize("precision,filler", [(0, (180_000,)), (0, (5,) * 250), (1, (350_000,))],
                         ids=["fp64", "fp64 many cells", "fp32_local"])
def test_narrow_quads_match_the_default_with_the_default_engine(gwcapi, gpu_ctx, precision, filler):
    batches = []
    for extra in (filler, ()):
        b = gwcapi.Batch(gpu_ctx, _cells(gwcapi, extra), precision=precision)
        b.set_mode(frozen=False, digest=False)
        for c, n in enumerate(SIZES):
            b.set_cru_state(c, **_state(n, n))
        assert b.running() == ((4, 64, 1) if extra else (4, 256, 1))
        b.step(60)
        batches.append(b)
    _same(*batches)
    for b in batches:
        b.close()


def test_replayed_graphs_of_the_one_lane_kernels_match_the_quads(gwcapi, gpu_ctx):
    a, b = _open(gwcapi, gpu_ctx, (340_000,)), _open(gwcapi, gpu_ctx, ())
    a.set_graph(16)
    assert a.running() == (1, 64, 2) and a.steps_per_launch() == 1 and b.running() == (4, 256, 1)
    for chunk in (40, 1, 75):
        a.step(chunk)
        b.step(chunk)
        _same(a, b)
    a.close()
    b.close()


UNIFORM = [
    (0, (4, 64, 1), 256, 1, (4, 64, 1)), (0, (4, 64, 1), 256, 15, (4, 64, 1)), (0, (4, 64, 1), 257, 17, (4, 64, 1)),
    (0, (4, 64, 1), 256, 65, (4, 64, 1)), (0, (4, 64, 1), 6, 57_001, (1, 64, 2)), (0, (4, 64, 1), 4, 240_001, (1, 64, 4)),
    (0, (4, 64, 1), 4, 650_001, (1, 64, 8)), (1, (4, 256, 1), 7, 50_003, (4, 64, 1)),
    (1, (1, 64, 4), 3, 100_001, (1, 64, 4)), (1, (1, 128, 2), 3, 100_001, (1, 128, 2)),
    (1, (1, 256, 4), 3, 100_001, (1, 256, 4)), (1, (1, 64, 8), 3, 100_001, (1, 64, 8))]


@pytest.mark.parametrize("precision,shape,cells,n,runs,steps_per_launch",
                         [u + (1,) for u in UNIFORM] + [u + (2,) for u in UNIFORM if u[4][:2] == (1, 64)])
def test_cells_of_one_size_match_a_mixed_batch(gwcapi, gpu_ctx, precision, shape, cells, n, runs, steps_per_launch):
    """Block ranges by arithmetic against the table, in the kernels of large batches."""
    g = gwcapi.default_globals()
    g.V, g.m, g.h, g.j = 10.0, 0.99, 1e-3, 0.1
    out = []
    for other in ((), (n + 3,)):
        b = gwcapi.Batch(gpu_ctx, [gwcapi.make_cell(k, 40 + c, None, _pace(gwcapi)) for c, k in enumerate((n,) * cells + other)],
                         precision=precision, globals_=g)
        b.set_mode(frozen=False, digest=False)
        b.set_launch(*shape)
        b.set_steps_per_launch(steps_per_launch)
        assert b.running() == runs and b.steps_per_launch() == steps_per_launch
        for chunk in (1, 2, 20):
            b.step(chunk)
        out.append(([x.as_array() for x in b.get_globals()][:cells], b.obs()[:cells],
                    [b.get_cru_state(c) for c in (0, 1, cells - 1)]))
        b.close()
    for x, y in zip(out[0][0], out[1][0]):
        assert np.array_equal(x, y)
    assert out[0][1] == out[1][1]
    for x, y in zip(out[0][2], out[1][2]):
        for k in KEYS:
            assert np.array_equal(x[k], y[k]), k


@pytest.mark.parametrize("shape,steps_per_launch", [((1, 64, 2), 1), ((1, 64, 4), 1), ((1, 64, 4), 2), ((1, 64, 8), 2),
                                                    ((1, 128, 4), 1), ((1, 256, 8), 1)])
def test_refilled_lanes_run_the_same_dynamics(gwcapi, gpu_ctx, shape, steps_per_launch):
    """FP32-local lanes that take several CRUs against one CRU per lane: the same
    state after the first step, whose constants come from the initial state
    alone; after 10 ms of a beat (upstroke and release) the same V within 1 mV and
    Cai within 5%, since only the rounding of the flux sums, and through it the
    odd event, differs; after 30 ms every channel count valid."""
    def start(extra, launch, spl):
        b = gwcapi.Batch(gpu_ctx, [gwcapi.make_cell(k, 40 + c, None, _pace(gwcapi))
                                   for c, k in enumerate((12_500, 12_500, 3001) + extra)], precision=1)
        b.set_mode(frozen=False, digest=False)
        b.set_launch(*launch)
        b.set_steps_per_launch(spl)
        return b

    a, b = start((300_000,), shape, steps_per_launch), start((), (1, 64, 1), 1)
    assert a.running() == shape and a.steps_per_launch() == steps_per_launch and b.running() == (1, 64, 1)
    for x in (a, b):
        x.step(1)
    for c in range(3):
        x, y = a.get_cru_state(c), b.get_cru_state(c)
        for k in KEYS:
            assert np.array_equal(x[k], y[k]), (c, k)
    for x in (a, b):
        x.step(9999)
    ga, gb = (np.array([g.as_array() for g in x.get_globals()[:3]]) for x in (a, b))
    dv, dca = np.abs(ga[:, 0] - gb[:, 0]), np.abs(ga[:, 3] - gb[:, 3]) / gb[:, 3]
    say(f"  {shape}: |dV| <= {dv.max():.3g} mV, |dCai|/Cai <= {dca.max():.3g}")
    assert np.all(dv < 1.0) and np.all(dca < 0.05)
    b.close()
    a.step(20_000)
    for c in range(4):
        s = a.get_cru_state(c)
        R = s["RyR"]
        assert np.all(R.sum(axis=2) == 5) and np.all(R[..., :2] >= 0)
        assert np.all(R[..., 2] + R[..., 3] >= 0) and np.all(R[..., 4] + R[..., 5] >= 0)
        assert np.all((s["LCC"] >= 1) & (s["LCC"] <= 12))
        open_lcc = ((s["LCC"] == 6) | (s["LCC"] == 12)) & (s["LCC_inactivation"] == 1)
        assert np.all(s["JLCC"][~open_lcc] == 0.0)
        assert np.all(np.isfinite(s["CaSS"])) and np.all(s["CaSS"] > 0) and np.all(s["CaJSR"] > 0)
    a.close()
