"""Velocities near the smallest double in the FP64 step.

Over a density that is a power of two a denormal momentum divides without a
remainder, so the checks of the shared reciprocal must look at the momenta
themselves.  Beside a cell of ordinary velocity such a velocity has a slope of its
own size, and half of that slope is rounded before it is added.  The result reaches
the arrays where nothing larger covers it: the cells hold no energy (their pressure
is the floor, their sound speed smallc), and gamma near 1 gives the energy's flux a
factor of a hundred.  Every array must equal the CPU oracle's bit for bit, on the
block kernel (tiles 1 and 16) and on the march (24 and 45).
"""
import numpy as np
import pytest

import oracle_lib as O
from euler2d_kokkos_amd import E2D_U, E2D_U2, HydroParams, HydroRun

pytestmark = pytest.mark.gpu

TINY = 2.0**-1074
MOMENTA = [0.0, -0.0, TINY, -TINY, 2 * TINY, 3 * TINY, -5 * TINY, 2.0**-1040, -(2.0**-1030),
           2.0**-1000, -(2.0**-968), 2.0**-903, -(2.0**-901), 2.0**-900, 3 * 2.0**-899]


def _params(slope, riemann, nx):
    return O.default_params(nx=nx, ny=45, ymax=45.0 / nx, gamma0=1.01, smallc=1.0, cfl=0.8,
                            nStepmax=2, tEnd=1e9, problemType=1, honor_riemann=1,
                            riemannSolverType=riemann, slope_type=slope)


def _state(p, density, axis, seed):
    """Along `axis`, groups of five cells with tiny velocities of that direction
    between groups of three cells at 1 or -1; no energy."""
    rng = np.random.default_rng(seed)
    a = np.zeros((p.isize, p.jsize, 4))
    shape = a.shape[:2]
    a[..., 0] = density
    place = np.arange(shape[axis]) % 8
    place = place[:, None] if axis == 0 else place[None, :]
    rare = rng.random(shape) < 0.25  # mostly the smallest
    m = np.asarray(MOMENTA)[rng.integers(0, np.where(rare, len(MOMENTA), 7))]
    a[..., 2 + axis] = np.where(place < 5, m, density * np.where(place == 6, -1.0, 1.0))
    return a


def _oracle(p, a):
    ora = O.OracleRun(p)
    for which in (0, 1):
        ora.set(which, a)
    ora.run()
    return ora


def _same(got, want, what):
    np.testing.assert_array_equal(got.view(np.int64), want.view(np.int64), err_msg=what)


@pytest.mark.parametrize("tile", [1, 16, 24, 45])
@pytest.mark.parametrize("riemann", [1, 2], ids=["hll", "hllc"])
@pytest.mark.parametrize("slope", [1.0, 2.0], ids=["minmod", "mc"])
@pytest.mark.parametrize("density", [1.0, 2.0, 0.5, 3.0])
@pytest.mark.parametrize("axis", [0, 1], ids=["x", "y"])
def test_tiny_velocities(gpu_available, axis, density, slope, riemann, tile):
    p = _params(slope, riemann, 128 if density >= 1.0 else 130)
    a = _state(p, density, axis, seed=5)
    ora = _oracle(p, a)
    run = HydroRun(HydroParams(p.copy()))
    run.set_tile(tile)
    run.set_state(E2D_U, a)
    run.set_state(E2D_U2, a)
    run.run()
    what = f"axis {axis} density {density} slope {slope} riemann {riemann} tile {tile}"
    assert (run.t, run.nStep) == (ora.t, ora.nStep), what
    for which in (E2D_U, E2D_U2):
        _same(run.get_state(which), ora.get(which), what)
