"""The state a batch is created in, sampled on the device with one lane per CRU:
cells whose sizes lie at the edges of its blocks, in one batch, against the same
sampler on the host. Every field is the same."""
import numpy as np
import pytest

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
