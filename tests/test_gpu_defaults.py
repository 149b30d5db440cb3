"""What a new run or batch chooses for itself: tile and launch mode."""
import pytest

import oracle_lib as O
from euler2d_kokkos_amd import (E2D_BATCH_LAUNCH_PERSISTENT, E2D_BATCH_LAUNCH_STEPS,
                                E2D_PRECISION_FP32_SPLIT, E2D_PRECISION_FP64, HydroParams, HydroRun)
from euler2d_kokkos_amd.batch import HydroBatch, make_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [E2D_PRECISION_FP64, E2D_PRECISION_FP32_SPLIT])
@pytest.mark.parametrize("n", [64, 300, 512])
def test_wide_addressing_takes_the_march_tile(gpu_available, monkeypatch, n, precision):
    """64-bit row offsets leave a small grid to the march, so its tile must be the
    march's: the one of a solver that the block kernel is not built for."""
    p = O.default_params(nx=n, ny=n, problemType=1, honor_riemann=1, riemannSolverType=0)
    with HydroRun(HydroParams(p.copy()), precision=precision) as run:
        march = run.get_tile()
    p.riemannSolverType = 2
    with HydroRun(HydroParams(p.copy()), precision=precision) as run:
        block = run.get_tile()
    assert block != march
    monkeypatch.setenv("E2D_WIDE_ADDRESSING", "1")
    with HydroRun(HydroParams(p.copy()), precision=precision) as run:
        assert run.get_tile() == march


@pytest.mark.parametrize("precision", [E2D_PRECISION_FP64, E2D_PRECISION_FP32_SPLIT])
def test_default_batch_launch_needs_enough_instances(gpu_available, precision):
    """Equal grids fill the queues evenly; the persistent launch is the default from
    12 a queue on.  The default tile is the launch mode's own, also after a later
    choice of the mode, until a tile is set."""
    def batch(count):
        ps = [make_params(nx=64, ny=64, problemType=1) for _ in range(count)]
        return HydroBatch(ps, precision=precision)

    b = batch(8)
    queues = b.queue_info()[0]
    b.close()
    few, many = batch(11 * queues), batch(12 * queues)
    assert few.queue_info() == (queues, 1.0) and many.queue_info() == (queues, 1.0)
    assert few.get_launch() == E2D_BATCH_LAUNCH_STEPS
    assert many.get_launch() == E2D_BATCH_LAUNCH_PERSISTENT
    many.close()
    steps = few.info()["waves"]
    few.set_launch(E2D_BATCH_LAUNCH_PERSISTENT)
    assert few.info()["waves"] == 11 * queues * 2 * 4  # 16 or 20 rows: two strips of four segments
    few.set_launch(E2D_BATCH_LAUNCH_STEPS)
    assert few.info()["waves"] == steps
    few.set_tile(64)
    for mode in (E2D_BATCH_LAUNCH_STEPS, E2D_BATCH_LAUNCH_PERSISTENT):
        few.set_launch(mode)
        assert few.info()["waves"] == 11 * queues * 2
    few.close()
