"""FP32-local shapes of several CRUs per lane: below 300,000 CRUs they run one
CRU per lane (the shape asked for is still reported), above it refilled lanes;
cells at the edges of their tiles, one and two steps per launch. Channel states
are those of one CRU per lane, and every launch of a batch gives the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = (1, 63, 64, 65, 255, 256, 257, 512, 513, 2049)
KEYS = ("CaSS", "CaJSR", "LCC", "LCC_inactivation", "RyR", "ClCh", "JLCC")


def _run(gwcapi, ctx, shape, steps_per_launch, filler):
    pace = {"kind": gwcapi.PROTO_PACE, "period": 500.0, "duration": 1.0, "amplitude": 100.0, "start": 0.0}
    g = gwcapi.default_globals()
    g.V, g.m, g.h, g.j = 10.0, 0.99, 1e-3, 0.1
    b = gwcapi.Batch(ctx, [gwcapi.make_cell(n, 90 + n, None, pace) for n in SIZES + filler], precision=1, globals_=g)
    b.set_mode(frozen=False, digest=False)
    b.set_launch(*shape)
    b.set_steps_per_launch(steps_per_launch)
    assert b.launch() == shape
    for chunk in (1, 2, 38):
        b.step(chunk)
    out = [b.get_cru_state(c) for c in range(len(SIZES))]
    b.close()
    return out


@pytest.mark.parametrize("filler", [(), (300_000,)], ids=["one per lane", "refilled"])
@pytest.mark.parametrize("threads,per_lane,steps_per_launch", [(64, 2, 1), (64, 4, 1), (64, 4, 2), (64, 8, 2), (128, 4, 1),
                                                               (256, 8, 1)])
def test_shapes_of_several_crus_per_lane(gwcapi, gpu_ctx, threads, per_lane, steps_per_launch, filler):
    one = _run(gwcapi, gpu_ctx, (1, threads, 1), 1, ())
    several = _run(gwcapi, gpu_ctx, (1, threads, per_lane), steps_per_launch, filler)
    again = _run(gwcapi, gpu_ctx, (1, threads, per_lane), steps_per_launch, filler)
    for c in range(len(SIZES)):
        for k in KEYS:
            assert np.array_equal(several[c][k], again[c][k]), (c, k)
            if several[c][k].dtype.kind != "f" or not filler:   # refilled lanes may round their sums differently
                assert np.array_equal(several[c][k], one[c][k]), (c, k)
