"""The state a batch is created in, sampled on the device with one lane per CRU:
cells whose sizes lie at the edges of its blocks, in one batch, against the same
sampler on the host. Every field is the same."""
import numpy as np
import pytest

from oracle.oracle import OracleModel

from .test_gpu_parity import assert_globals_equal, assert_states_equal

pytestmark = pytest.mark.gpu

SIZES = (1, 3, 63, 64, 65, 255, 256, 257, 513, 1250)


@pytest.mark.parametrize("prng", range(6))
@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32_local"])
def test_initial_state_matches_the_host_sampler(gwcapi, gpu_ctx, prng, precision):
    b = gwcapi.Batch(gpu_ctx, [gwcapi.make_cell(n, 70 + n) for n in SIZES], precision=precision, prng=prng)
    for c, n in enumerate(SIZES):
        want, got = gwcapi.rest_state(n, 70 + n, prng), b.get_cru_state(c)
        for k in want:
            assert np.array_equal(want[k], got[k]), (n, k)
    b.close()


@pytest.mark.parametrize("n", [1, 255, 256, 257, 1023, 1024, 1025, 2049])
def test_first_steps_match_the_oracle(gwcapi, gpu_ctx, n):
    """The sums the first steps start from, of cells at the edges of the block that forms them."""
    b = gwcapi.Batch(gpu_ctx, [gwcapi.make_cell(n, 11)])
    m = OracleModel(n, seed=11)
    m.sample_rest_state()
    for _ in range(3):
        b.step(1)
        assert m.step(1e-3, 0.0) == 0
        assert_globals_equal(b.get_globals()[0], m.globals())
    assert_states_equal(b.get_cru_state(0), m.state())
    b.close()
