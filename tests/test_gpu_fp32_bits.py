"""The bits of FP32-local results do not follow the compiler: which products are
fused is written out in the source, per layout. Subspace Ca on both sides of both
lumping thresholds with RyRs in every state, so that every form of the rates is
taken; the expected sums are those of an earlier build, whose compiler had arranged
them so. (The FP64 form is compared with the oracle instead.)"""
import hashlib

import numpy as np
import pytest

from .test_gpu_lane64 import _state

pytestmark = pytest.mark.gpu

SIZES = (700, 64, 1250)
KEYS = ("CaSS", "CaJSR", "LCC", "LCC_inactivation", "RyR", "ClCh", "JLCC")
QUADS, LANES = "a2bfa3c8506b611da5ca535fdc74977e75c257ea", "9c90da7bffdef5f57ab44a3431e467cd4523495f"


def _sum(gwcapi, ctx, shape, steps_per_launch, filler):
    pace = {"kind": gwcapi.PROTO_PACE, "period": 500.0, "duration": 1.0, "amplitude": 100.0, "start": 0.0}
    g = gwcapi.default_globals()
    g.V, g.m, g.h, g.j = 10.0, 0.99, 1e-3, 0.1
    cells = [gwcapi.make_cell(n, 500 + n, None, pace) for n in SIZES + filler]
    for d in cells:   # rates of the pair (5,6) that are a large part of the total
        d.params.k52, d.params.k65, d.params.k43 = 333.3, 41.7, 51.3
    b = gwcapi.Batch(ctx, cells, precision=1, globals_=g)
    b.set_mode(frozen=False, digest=False)
    b.set_launch(*shape)
    b.set_steps_per_launch(steps_per_launch)
    for c, n in enumerate(SIZES):
        st = _state(n, n)
        st["CaSS"][::2] = np.random.default_rng(n).uniform(4e-5, 1.1e-4, st["CaSS"][::2].shape)
        b.set_cru_state(c, **st)
    b.step(400)
    m = hashlib.sha1()
    for c in range(len(SIZES)):
        s = b.get_cru_state(c)
        m.update(b.get_globals()[c].as_array().tobytes())
        for k in KEYS:
            m.update(np.ascontiguousarray(s[k]).tobytes())
    b.close()
    return m.hexdigest()


@pytest.mark.parametrize("shape,steps_per_launch,filler,want", [
    ((4, 256, 1), 1, (), QUADS), ((4, 64, 1), 1, (350_000,), QUADS),
    ((1, 64, 1), 1, (), LANES), ((1, 256, 1), 1, (), LANES), ((1, 64, 1), 2, (), LANES),
    ((1, 64, 4), 2, (300_000,), LANES), ((1, 128, 4), 1, (300_000,), LANES)])
def test_fp32_local_bits(gwcapi, gpu_ctx, shape, steps_per_launch, filler, want):
    assert _sum(gwcapi, gpu_ctx, shape, steps_per_launch, filler) == want
