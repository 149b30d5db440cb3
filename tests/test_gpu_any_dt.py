"""godunov_unsplit with time steps of either sign and any size: the checked FP64 forms
hold for |dt / dx| up to 2^40 only.  Block kernel (tile 7) and march (24), the state
after one and after two steps bit for bit against the CPU oracle, NaN for NaN.
"""
import numpy as np
import pytest

import oracle_lib as O
import test_gpu_bounded as B
from euler2d_kokkos_amd import E2D_U, E2D_U2, HydroParams, HydroRun

pytestmark = pytest.mark.gpu

STEPS = [0.0, 1e-3, 2.0**33, 1e20, 1e60, 1e110, 1e155, 1e300, np.inf]  # dx is about 2^-7


@pytest.mark.parametrize("tile", [7, 24])
@pytest.mark.parametrize("riemann", [1, 2], ids=["hll", "hllc"])
@pytest.mark.parametrize("slope", [1.0, 2.0], ids=["minmod", "mc"])
@pytest.mark.parametrize("dt", [s * v for v in STEPS for s in (1, -1)] + [np.nan])
def test_any_time_step(gpu_available, dt, slope, riemann, tile):
    p = O.default_params(**dict(B.BASE, nx=128 if slope == 1.0 else 130, riemannSolverType=riemann,
                                slope_type=slope))
    ora, a = B._state(p, "rest", seed=21)
    rng = np.random.default_rng(22)
    a[..., 2] = 0.3 * rng.normal(size=a.shape[:2])
    a[..., 3] = 0.3 * rng.normal(size=a.shape[:2])
    run = HydroRun(HydroParams(p.copy()))
    run.set_tile(tile)
    for which in (E2D_U, E2D_U2):
        ora.set(which, a)
        run.set_state(which, a)
    for n in range(2):
        ora.godunov_unsplit(n, dt)
        run.godunov_unsplit(n, dt)
        which = E2D_U2 if n == 0 else E2D_U
        g, o = run.get_state(which), ora.get(which)
        nan = np.isnan(o)
        what = f"step {n} dt {dt} slope {slope} riemann {riemann} tile {tile}"
        np.testing.assert_array_equal(np.isnan(g), nan, err_msg=what)
        np.testing.assert_array_equal(g.view(np.int64)[~nan], o.view(np.int64)[~nan], err_msg=what)
