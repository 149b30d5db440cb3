"""What a new run chooses for itself."""
import pytest

import oracle_lib as O
from euler2d_kokkos_amd import (E2D_PRECISION_FP32_SPLIT, E2D_PRECISION_FP64, HydroParams,
                                HydroRun)

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
