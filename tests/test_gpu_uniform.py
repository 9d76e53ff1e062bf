"""Batches whose cells have one size find a block's cell and CRUs by arithmetic,
others in a table: the same three cells, in a batch of their own and in one with
a fourth cell of another size, at the edges of the blocks of every kind of
launch shape. Every bit of both is the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = ("CaSS", "CaJSR", "LCC", "LCC_inactivation", "RyR", "ClCh", "JLCC")


@pytest.mark.parametrize("precision,shape", [(0, (4, 256, 1)), (0, (4, 64, 1)), (0, (4, 128, 4)), (1, (4, 256, 1)),
                                             (1, (1, 64, 1)), (1, (1, 256, 4)), (1, (1, 64, 8))])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 1250])
def test_cells_of_one_size_match_a_mixed_batch(gwcapi, gpu_ctx, n, precision, shape):
    pace = {"kind": gwcapi.PROTO_PACE, "period": 500.0, "duration": 1.0, "amplitude": 100.0, "start": 0.0}
    g = gwcapi.default_globals()
    g.V, g.m, g.h, g.j = 10.0, 0.99, 1e-3, 0.1
    batches = []
    for other in ((), (n + 3,)):
        cells = [gwcapi.make_cell(k, 40 + c, None, pace) for c, k in enumerate((n, n, n) + other)]
        b = gwcapi.Batch(gpu_ctx, cells, precision=precision, globals_=g)
        b.set_mode(frozen=False, digest=False)
        b.set_launch(*shape)
        for chunk in (1, 2, 47):
            b.step(chunk)
        batches.append(b)
    a, b = batches
    for c in range(3):
        assert np.array_equal(a.get_globals()[c].as_array(), b.get_globals()[c].as_array()), c
        sa, sb = a.get_cru_state(c), b.get_cru_state(c)
        for k in KEYS:
            assert np.array_equal(sa[k], sb[k]), (c, k)
        assert a.obs()[c] == b.obs()[c], c
    a.close()
    b.close()
