"""CRU state read and written in pieces of 65,536 CRUs: cells at the edges of a
piece, of odd size and of several pieces, in both precisions. What was set is
read back, whole and reduced, and the records of a run are the states a batch
of the same cell passes through."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PIECE = 65536
KEYS = ("CaSS", "CaJSR", "LCC", "LCC_inactivation", "RyR", "ClCh", "JLCC")


def _state(n, seed):
    rng = np.random.default_rng(seed)
    ryr = np.zeros((n, 4, 6), np.int32)
    for k in rng.integers(0, 6, size=(5, n, 4)):
        np.add.at(ryr, (*np.indices((n, 4)), k), 1)
    return {"CaSS": np.exp(rng.uniform(np.log(5e-5), np.log(0.1), (n, 4))), "CaJSR": rng.uniform(0.2, 0.9, n),
            "LCC": rng.integers(1, 13, (n, 4)), "LCC_inactivation": rng.integers(0, 2, (n, 4)), "RyR": ryr,
            "ClCh": rng.integers(0, 2, (n, 4)), "JLCC": rng.uniform(-1.0, 1.0, (n, 4))}


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32_local"])
@pytest.mark.parametrize("n", [1, 127, PIECE - 1, PIECE, PIECE + 1, 2 * PIECE + 129])
def test_state_goes_in_and_out_in_pieces(gwcapi, gpu_ctx, n, precision):
    b = gwcapi.Batch(gpu_ctx, [gwcapi.make_cell(m, 5 + m) for m in (3, n, 65)], precision=precision)
    want = _state(n, n)
    b.set_cru_state(1, **want)
    if precision:
        want["JLCC"] = want["JLCC"].astype(np.float32).astype(np.float64)
    got = b.get_cru_state(1)
    for k in KEYS:
        assert np.array_equal(got[k], want[k]), k
    red = b.get_cru_state_reduced(1)
    for k in ("CaSS", "CaJSR"):
        assert np.array_equal(red[k], want[k].astype(np.float32)), k
    for k in ("LCC", "LCC_inactivation", "ClCh"):
        assert np.array_equal(red[k].astype(np.int32), want[k]), k
    assert np.array_equal(red["RyR"], (want["RyR"][..., :5] * 6 ** np.arange(5)).sum(-1))
    for c, m in ((0, 3), (2, 65)):   # the neighbours are as they were made
        rest, got = gwcapi.rest_state(m, 5 + m), b.get_cru_state(c)
        for k in KEYS:
            assert np.array_equal(got[k], rest[k]), (c, k)
    b.close()


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32_local"])
@pytest.mark.parametrize("n,every", [(65, 1), (PIECE + 1, 3), (2 * PIECE + 129, 2)])
def test_records_are_the_states_a_batch_passes_through(gwcapi, gpu_ctx, n, every, precision):
    steps = 10
    crus = gwcapi.rest_state(n, 8)
    crus.update({k: v for k, v in _state(n, 9).items() if k in ("LCC", "RyR")})
    rec = gwcapi.run(gpu_ctx, gwcapi.Params.default(), n, 1e-3, steps, np.full(steps, 100.0), every, None, crus, 8, 0,
                     precision)
    b = gwcapi.Batch(gpu_ctx, [gwcapi.make_cell(n, 8)], precision=precision)
    b.set_mode(frozen=False, digest=False)
    b.set_cru_state(0, **{k: crus[k] for k in KEYS[:-1]})
    b.set_stimulus_table(0, np.full(steps, 100.0))
    done = 0
    for k, i in enumerate(range(0, steps, every)):
        b.step(i + 1 - done)
        done = i + 1
        got = b.get_cru_state(0)
        for key in KEYS[:-1]:
            assert np.array_equal(rec[key][k], got[key]), (k, key)
        assert rec["V"][k] == b.get_globals()[0].V
        assert rec["t"][k] == b.time()[0]
    b.close()
