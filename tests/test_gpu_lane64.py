"""FP64 batches large enough for the one-lane kernels (one lane per CRU, 2, 4
or 8 CRUs per lane, one or two Euler steps per launch, events of a wave applied
together): cells whose sizes lie at the edges of their tiles, in a batch with a
cell large enough to choose those kernels, against the same cells in a batch of
their own, which runs the quads. Every bit of both is the same."""
import numpy as np
import pytest

from .test_gpu_parity import say

pytestmark = pytest.mark.gpu

SIZES = (1, 63, 64, 65, 255, 256, 257, 511, 512, 513, 1250)
KEYS = ("CaSS", "CaJSR", "LCC", "LCC_inactivation", "RyR", "ClCh", "JLCC")


def _cells(gwcapi, filler):
    pace = {"kind": gwcapi.PROTO_PACE, "period": 500.0, "duration": 1.0, "amplitude": 100.0, "start": 0.0}
    return [gwcapi.make_cell(n, 300 + n, None, pace) for n in SIZES + filler]


def _state(n, seed):
    """Channels in every state and CaSS on both sides of both lumping thresholds."""
    rng = np.random.default_rng(seed)
    ryr = np.zeros((n, 4, 6), np.int32)
    for k in rng.integers(0, 6, size=(5, n, 4)):
        np.add.at(ryr, (*np.indices((n, 4)), k), 1)
    return {"CaSS": np.exp(rng.uniform(np.log(5e-5), np.log(0.1), (n, 4))), "CaJSR": rng.uniform(0.2, 0.9, n),
            "LCC": rng.integers(1, 13, (n, 4)), "LCC_inactivation": rng.integers(0, 2, (n, 4)), "RyR": ryr,
            "ClCh": rng.integers(0, 2, (n, 4))}


def _open(gwcapi, ctx, filler, prng=0):
    g = gwcapi.default_globals()
    g.V, g.m, g.h, g.j = 10.0, 0.99, 1e-3, 0.1
    b = gwcapi.Batch(ctx, _cells(gwcapi, filler), prng=prng, globals_=g)
    b.set_mode(frozen=False, digest=False)
    for c, n in enumerate(SIZES):
        b.set_cru_state(c, **_state(n, n))
    return b


def _same(a, b, observables=True):
    for c in range(len(SIZES)):
        x, y = a.get_globals()[c].as_array(), b.get_globals()[c].as_array()
        assert np.array_equal(x, y, equal_nan=True), c
        sx, sy = a.get_cru_state(c), b.get_cru_state(c)
        for k in KEYS:
            assert np.array_equal(sx[k], sy[k], equal_nan=sx[k].dtype.kind == "f"), (c, k)
        assert not observables or a.obs()[c] == b.obs()[c], c


@pytest.mark.parametrize("filler", [(640_000,), (1 << 20,), (1 << 20, 1 << 20, 500_000)],
                         ids=["2 per lane", "4 per lane", "8 per lane"])
@pytest.mark.parametrize("steps_per_launch", [0, 1])
def test_one_lane_kernels_match_the_quads(gwcapi, gpu_ctx, filler, steps_per_launch):
    a, b = _open(gwcapi, gpu_ctx, filler), _open(gwcapi, gpu_ctx, ())
    a.set_steps_per_launch(steps_per_launch)
    assert a.steps_per_launch() == (1 if steps_per_launch == 1 else 2)
    assert b.steps_per_launch() == 1
    for chunk in (1, 2, 57, 240):   # odd and even calls
        a.step(chunk)
        b.step(chunk)
        say(f"  {chunk} steps")
        _same(a, b)
    a.close()
    b.close()


def test_a_failing_cell_stops_at_the_same_step(gwcapi, gpu_ctx):
    """A NaN voltage: the cell stops with its status after the same SSA steps, the others go on."""
    a, b = _open(gwcapi, gpu_ctx, (640_000,)), _open(gwcapi, gpu_ctx, ())
    for x in (a, b):
        x.step(31)
        g = x.get_globals()[3]
        g.V = float("nan")
        x.set_globals(3, g)
        with pytest.raises(gwcapi.GwError) as e:
            x.step(40)
        assert "cell 3" in str(e.value)
    for c in range(len(SIZES)):
        assert np.array_equal(a.get_globals()[c].as_array(), b.get_globals()[c].as_array(), equal_nan=True), c
        sx, sy = a.get_cru_state(c), b.get_cru_state(c)
        for k in KEYS:
            assert np.array_equal(sx[k], sy[k], equal_nan=sx[k].dtype.kind == "f"), (c, k)
    a.close()
    b.close()


@pytest.mark.parametrize("ca", [0.0, 1e-320, -2e-5, 1e31], ids=["zero", "denormal", "negative", "huge"])
@pytest.mark.parametrize("constant", [None, 1e-40], ids=["constants of the model", "tiny KBSR"])
def test_quotients_that_need_scaling_match_the_quads(gwcapi, gpu_ctx, ca, constant):
    """A wave divides without scaling only where every operand allows it: one CRU of a cell, or one
    constant of all, outside that range."""
    def start(filler):
        cells = _cells(gwcapi, filler)
        for d in cells:
            if constant:
                d.params.KBSR = constant
        g = gwcapi.default_globals()
        g.V, g.m, g.h, g.j = 10.0, 0.99, 1e-3, 0.1
        b = gwcapi.Batch(gpu_ctx, cells, globals_=g)
        b.set_mode(frozen=False, digest=False)
        for c, n in enumerate(SIZES):
            st = _state(n, n)
            st["CaSS"][n // 2, 1] = ca
            b.set_cru_state(c, **st)
        try:
            b.step(3)
        except gwcapi.GwError as e:   # a concentration this large leaves the range of the fluxes
            assert ca > 1.0, e
        return b

    _same(start((640_000,)), start(()), observables=ca < 1.0)   # a cell that fails has NaN among its observables


@pytest.mark.parametrize("size,steps_per_launch", [(60, 1), (64, 2)])
def test_cells_smaller_than_a_wave_stay_with_the_quads(gwcapi, gpu_ctx, size, steps_per_launch):
    b = gwcapi.Batch(gpu_ctx, [gwcapi.make_cell(size, c) for c in range(6000)])
    b.set_mode(frozen=False, digest=False)
    assert b.steps_per_launch() == steps_per_launch
    b.step(5)
    b.close()


@pytest.mark.parametrize("prng", range(1, 6))
@pytest.mark.parametrize("filler", [(340_000,), (1 << 20,), (1 << 20, 1 << 20, 500_000)],
                         ids=["2 per lane", "4 per lane", "8 per lane"])
def test_one_lane_kernels_match_the_quads_with_every_engine(gwcapi, gpu_ctx, prng, filler):
    a, b = _open(gwcapi, gpu_ctx, filler, prng), _open(gwcapi, gpu_ctx, (), prng)
    assert a.steps_per_launch() == 2
    for steps_per_launch, chunk in ((0, 21), (1, 20)):
        a.set_steps_per_launch(steps_per_launch)
        a.step(chunk)
        b.step(chunk)
        _same(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("prng", range(1, 6))
@pytest.mark.parametrize("precision,filler", [(0, 180_000), (1, 350_000)], ids=["fp64", "fp32_local"])
def test_narrow_quads_match_the_default_with_every_engine(gwcapi, gpu_ctx, prng, precision, filler):
    """The quads of large batches (64 threads) against those of small ones (256)."""
    batches = []
    for extra in ((filler,), ()):
        b = gwcapi.Batch(gpu_ctx, _cells(gwcapi, extra), precision=precision, prng=prng)
        b.set_mode(frozen=False, digest=False)
        for c, n in enumerate(SIZES):
            b.set_cru_state(c, **_state(n, n))
        b.step(25)
        batches.append(b)
    _same(*batches)
    for b in batches:
        b.close()
