"""Cells whose sound speed is infinite or no number: energies near the largest double,
also such that only gamma p / rho overflows, infinities and NaN in each variable.  The wave speeds take the short
square root in FP64, which has no infinity of its own; block kernel (tile 7) and march (24),
bit for bit against the CPU oracle, NaN for NaN.
"""
import numpy as np
import pytest

import oracle_lib as O
import test_gpu_bounded as B
from euler2d_kokkos_amd import E2D_U, E2D_U2, HydroParams, HydroRun

pytestmark = pytest.mark.gpu

CELLS = {  # density, energy, momentum
    "speed only": (1e-3, 1e304, 0.0),  # at gamma 16
    "speed only in part": (1.0, 3e307, 0.0),
    "overflow": (1e-3, 1e308, 0.0),
    "sum": (1.0, 1.7e308, 0.0),
    "energy": (1.0, np.inf, 0.0),
    "negative": (1.0, -np.inf, 0.0),
    "density": (np.inf, 1.0, 0.0),
    "momentum": (1.0, 2.5, np.inf),
    "nan": (1.0, np.nan, 0.1),
    "nan momentum": (1.0, 2.5, np.nan),
    "largest speed": (1.0, 1e307, 1e150),
}


@pytest.mark.parametrize("tile", [7, 24])
@pytest.mark.parametrize("riemann", [1, 2], ids=["hll", "hllc"])
@pytest.mark.parametrize("slope", [1.0, 2.0], ids=["minmod", "mc"])
@pytest.mark.parametrize("cell", sorted(CELLS))
def test_infinite_sound_speed(gpu_available, cell, slope, riemann, tile):
    p = O.default_params(**dict(B.BASE, nx=128 if slope == 1.0 else 130, riemannSolverType=riemann,
                                slope_type=slope, nStepmax=3,
                                gamma0=16.0 if "speed only" in cell else 1.4))
    ora, a = B._state(p, "rest", seed=11)
    rng = np.random.default_rng(12)
    a[..., 2] = 0.3 * rng.normal(size=a.shape[:2])
    a[..., 3] = 0.3 * rng.normal(size=a.shape[:2])
    rho, energy, mom = CELLS[cell]
    for i, j in ((31, 20), (32, 20), (90, 8), (64, 40)):
        a[i, j] = rho, energy, mom, -mom
    with np.errstate(all="ignore"):
        for which in (0, 1):
            ora.set(which, a)
        ora.run()
    run = HydroRun(HydroParams(p.copy()))
    run.set_tile(tile)
    run.set_state(E2D_U, a)
    run.set_state(E2D_U2, a)
    run.run()
    B._same_bits(run, ora, f"{cell} slope {slope} riemann {riemann} tile {tile}")
