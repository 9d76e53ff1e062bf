"""The configuration a batch's steps run in, which the shape asked for is a
request for: on both sides of every line of the rule."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,asked,cells,crus,runs", [
    (0, (4, 256, 1), 1, 12_500, (4, 256, 1)),
    (0, (4, 512, 1), 1, 12_500, (4, 256, 1)),
    (0, (4, 64, 1), 1, 179_999, (4, 256, 1)),
    (0, (4, 256, 1), 1, 180_000, (4, 64, 1)),
    (0, (4, 256, 1), 255, 10, (4, 256, 1)),
    (0, (4, 256, 1), 256, 10, (4, 64, 1)),
    (0, (4, 256, 1), 1, 339_999, (4, 64, 1)),
    (0, (4, 256, 1), 1, 340_000, (1, 64, 2)),
    (0, (4, 128, 4), 1, 339_999, (4, 128, 4)),
    (0, (4, 128, 4), 1, 340_000, (1, 64, 2)),
    (0, (4, 64, 1), 2, 474_999, (1, 64, 2)),
    (0, (4, 64, 1), 2, 475_000, (1, 64, 4)),
    (0, (4, 64, 1), 4, 624_999, (1, 64, 4)),
    (0, (4, 64, 1), 4, 625_000, (1, 64, 8)),
    (0, (4, 256, 1), 6000, 63, (4, 64, 1)),
    (1, (4, 64, 1), 1, 349_999, (4, 256, 1)),
    (1, (4, 128, 1), 1, 350_000, (4, 64, 1)),
    (1, (1, 128, 4), 1, 299_999, (1, 128, 1)),
    (1, (1, 128, 4), 1, 300_000, (1, 128, 4)),
    (1, (1, 64, 1), 1, 1000, (1, 64, 1)),
])
def test_the_configuration_that_runs(gwcapi, gpu_ctx, precision, asked, cells, crus, runs):
    b = gwcapi.Batch(gpu_ctx, [gwcapi.make_cell(crus, c) for c in range(cells)], precision=precision)
    b.set_mode(frozen=False, digest=False)
    b.set_launch(*asked)
    assert b.launch() == asked and b.running() == runs
    if precision == 0:
        b.set_mode(frozen=False, digest=True)   # digests are kept by the quads of 256 threads
        assert b.running() == (4, 256, 1)
    b.close()


@pytest.mark.parametrize("precision,cells,alike", [
    (0, (2000, 300), [("4x64", "4x128", "4x256", "4x512")]),
    (0, (340_000,), [("4x64", "4x256", "4x64x2", "4x256x4")]),
    (1, (2000, 300), [("4x64", "4x128", "4x256", "4x512"), ("1x64", "1x64x2", "1x64x8"), ("1x256", "1x256x4")]),
    (1, (300_000,), [("4x64", "4x512")])], ids=["fp64", "fp64 large", "fp32_local", "fp32_local refilled"])
def test_the_autotuner_times_shapes_that_run_alike_once(gwcapi, gpu_ctx, precision, cells, alike):
    b = gwcapi.Batch(gpu_ctx, [gwcapi.make_cell(n, n) for n in cells], precision=precision)
    b.set_mode(frozen=False, digest=False)
    b.step(10)
    shape, ms = b.autotune(20)
    for names in alike:
        assert len({ms[k] for k in names}) == 1 and ms[names[0]] > 0, ms
    assert b.launch() == shape
    assert b.running() == shape or (precision == 0 and cells == (340_000,))   # no quad shape runs as itself there
    if precision and cells == (300_000,):
        assert len({ms[k] for k in ("1x64", "1x64x2", "1x64x4", "1x64x8")}) > 1   # these are kernels of their own
    b.close()
