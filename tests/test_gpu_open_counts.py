"""Subunits with more open RyRs than a signed byte holds (the two open counts of
a subunit are accepted up to 100 each): the one-lane kernels against the quads
in FP64, their release flux against FP64 in the FP32-local form, and the sum of
a lane that runs nearly all CRUs of its wave."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = ("CaSS", "CaJSR", "LCC", "LCC_inactivation", "RyR", "ClCh", "JLCC")


def _state(n, ca, ryr):
    return {"CaSS": np.broadcast_to(ca, (n, 4)), "CaJSR": np.full(n, 0.9), "LCC": np.ones((n, 4)),
            "LCC_inactivation": np.ones((n, 4)), "RyR": np.broadcast_to(ryr, (n, 4, 6)), "ClCh": np.zeros((n, 4))}


@pytest.mark.parametrize("filler", [(340_000,), (1 << 20,)], ids=["2 per lane", "4 per lane"])
@pytest.mark.parametrize("steps_per_launch", [0, 1])
def test_fp64_lanes_match_the_quads(gwcapi, gpu_ctx, filler, steps_per_launch):
    sizes = (1, 65, 300)
    batches = []
    for extra in (filler, ()):
        cells = [gwcapi.make_cell(n, 7 + n) for n in sizes + extra]
        for c in cells:
            c.params.rRyR = 0.02
        b = gwcapi.Batch(gpu_ctx, cells)
        b.set_mode(frozen=False, digest=False)
        b.set_steps_per_launch(steps_per_launch)
        for c, n in enumerate(sizes):
            rng = np.random.default_rng(n)
            ryr = np.concatenate([rng.integers(0, 6, (n, 4, 2)), rng.integers(70, 101, (n, 4, 2)), rng.integers(0, 6, (n, 4, 2))], 2)
            b.set_cru_state(c, **_state(n, np.exp(rng.uniform(np.log(5e-5), np.log(3e-3), (n, 4))), ryr))
        batches.append(b)
    a, b = batches
    for chunk in (1, 2, 5):
        a.step(chunk)
        b.step(chunk)
        for c in range(len(sizes)):
            x, y = a.get_cru_state(c), b.get_cru_state(c)
            for k in KEYS:
                assert np.array_equal(x[k], y[k]), (c, k)
            assert np.array_equal(a.get_globals()[c].as_array(), b.get_globals()[c].as_array()), c
            assert a.obs()[c] == b.obs()[c], c
    assert x["RyR"][..., 2:4].sum(2).max() > 127
    a.close()
    b.close()


@pytest.mark.parametrize("shape,steps_per_launch,filler", [((1, 64, 1), 1, ()), ((1, 64, 1), 2, ()), ((1, 64, 4), 2, (300_000,))],
                         ids=["one step", "two steps", "refilled"])
def test_fp32_lanes_release_as_fp64_does(gwcapi, gpu_ctx, shape, steps_per_launch, filler):
    """200 open RyRs stay open while others go to and fro, each time with the
    release flux formed again: it is rRyR x 200 x (CaJSR - CaSS), CaSS below 1% of
    CaJSR, so the two forms' integrals differ by less than 2%."""
    def release(precision, extra):
        cells = [gwcapi.make_cell(n, 3) for n in (200,) + extra]
        p = cells[0].params
        p.rRyR, p.k12, p.k21 = 0.02, 1e12, 1e4
        p.k23 = p.k25 = p.k32 = p.k34 = p.k43 = p.k45 = 0.0
        b = gwcapi.Batch(gpu_ctx, cells, precision=precision)
        b.set_mode(frozen=False, digest=False)
        if precision:
            b.set_launch(*shape)
            b.set_steps_per_launch(steps_per_launch)
        b.set_cru_state(0, **_state(200, 1e-4, [5, 0, 100, 100, 0, 0]))
        b.step(20)
        assert np.all(b.get_cru_state(0)["RyR"][..., 2:4] == 100) and b.get_cru_state(0)["CaSS"].max() < 9e-3
        o = b.obs()[0]
        b.close()
        return o["int_Jrel"], o["sum_open_RyR_frac"]

    (want, want_open), (got, got_open) = release(0, ()), release(1, filler)
    assert got_open == want_open == 20 * 40.0
    assert want > 0 and abs(got - want) < 0.02 * want


def test_a_lane_that_runs_nearly_every_cru_of_its_wave(gwcapi, gpu_ctx):
    """Lanes 1 to 63 hold a CRU whose chloride channels flip 2e4 times in the step,
    so lane 0 takes the other 449 CRUs of the wave, with 800 open RyRs each."""
    n = 512
    cells = [gwcapi.make_cell(k, 5) for k in (n, 300_000)]
    p = cells[0].params
    p.rRyR = p.k12 = p.k23 = p.k25 = p.k32 = p.k34 = p.k45 = 0.0
    p.k43 = 1.0
    p.kfClCh = p.kbClCh = 1e7
    b = gwcapi.Batch(gpu_ctx, cells, precision=1)
    b.set_mode(frozen=False, digest=False)
    b.set_launch(1, 64, 8)
    slow = (np.arange(n) >= 1) & (np.arange(n) < 64)
    b.set_cru_state(0, **_state(n, np.where(slow, 1.0, 1e-9)[:, None],
                                np.where(slow[:, None, None], [5, 0, 0, 0, 0, 0], [0, 0, 100, 100, 0, 0])))
    i0 = b.iterations()
    b.step(1)
    assert b.iterations() - i0 > 300_000 + 63 * 10_000
    assert b.get_cru_state(0)["RyR"][..., 2:4].sum() == 449 * 800
    assert b.obs()[0]["sum_open_RyR_frac"] == 449 * 800 / (20.0 * n)
    b.close()
