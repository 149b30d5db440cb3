"""The limits of the bounded FP64 quotients: the largest and smallest values that
they are used for, and the smallest floors and extreme gammas of the decks that get
them.  A few cells on either side of each limit in a smooth state, and states near
floors on either side of theirs; block kernel (tile 7) and march (24), bit for bit
against the CPU oracle.
"""
import numpy as np
import pytest

import oracle_lib as O
import test_gpu_bounded as B
import test_gpu_rate as R
from euler2d_kokkos_amd import E2D_U, E2D_U2, HydroParams, HydroRun

pytestmark = pytest.mark.gpu

# density 2^80, pressure 2^160 (about 0.6 of the energy), velocity ~2^60.5, momenta 2^-801
LIMITS = {
    "density": ("rho", [2.0**80, 2.0**80 * (1 + 2.0**-52), 2.0**81, 1e30]),
    "pressure": ("energy", [2.0**160, 2.0**161, 3.3e48, 1e52]),
    "velocity": ("mom", [2.0**60, -2.0**60.5, 2.0**61, 1.7e18]),
    "tiny": ("mom", [0.0, -0.0, 2.0**-801, -2.0**-801 * (1 - 2.0**-53), 2.0**-800, -2.0**-850]),
}


def _check(p, a, tile, what):
    ora = O.OracleRun(p)
    for which in (0, 1):
        ora.set(which, a)
    ora.run()
    run = HydroRun(HydroParams(p.copy()))
    run.set_tile(tile)
    run.set_state(E2D_U, a)
    run.set_state(E2D_U2, a)
    run.run()
    B._same_bits(run, ora, what)


@pytest.mark.parametrize("tile", [7, 24])
@pytest.mark.parametrize("riemann", [1, 2], ids=["hll", "hllc"])
@pytest.mark.parametrize("slope", [1.0, 2.0], ids=["minmod", "mc"])
@pytest.mark.parametrize("edge", sorted(LIMITS))
def test_values_at_the_limits(gpu_available, monkeypatch, edge, slope, riemann, tile):
    monkeypatch.setitem(B.EDGES, edge, LIMITS[edge])
    p = O.default_params(**dict(B.BASE, nx=128 if slope == 1.0 else 130, riemannSolverType=riemann,
                                slope_type=slope))
    _, a = B._state(p, edge, seed=7)
    _check(p, a, tile, f"{edge} slope {slope} riemann {riemann} tile {tile}")


FLOORS = {  # smallr, smallc
    "lowest": (2.0**-110, 2.0**-110),
    "below in density": (2.0**-111, 2.0**-110),
    "below in speed": (2.0**-110, 2.0**-111),
    "usual": (1e-10, 1e-10),
    "interstellar": (1e-30, 1e-3),
}


@pytest.mark.parametrize("tile", [7, 24])
@pytest.mark.parametrize("riemann", [1, 2], ids=["hll", "hllc"])
@pytest.mark.parametrize("gamma", [1 + 2.0**-20, 5.0 / 3.0, 16.0])
@pytest.mark.parametrize("thin", [False, True], ids=["ordinary", "thin"])
@pytest.mark.parametrize("floors", sorted(FLOORS))
def test_states_at_the_floors(gpu_available, floors, thin, gamma, riemann, tile):
    """Densities of order one, or a few times the floor; among them cells at the floors
    of density and pressure, cells without energy or with a negative one, and cells
    at rest."""
    smallr, smallc = FLOORS[floors]
    p = O.default_params(**dict(B.BASE, nx=128 if thin else 130, riemannSolverType=riemann,
                                gamma0=gamma, smallr=smallr, smallc=smallc, cfl=0.3))
    rng = np.random.default_rng(17)
    shape = (p.isize, p.jsize)
    pick = rng.random(shape)
    rho = np.exp(0.3 * rng.normal(size=shape)) * (8 * smallr if thin else 1.0)
    rho = np.where((pick > 0.2) & (pick < 0.23), smallr, rho)
    u, v = 0.5 * rng.normal(size=shape), 0.5 * rng.normal(size=shape)
    e = np.exp(0.3 * rng.normal(size=shape)) * max(1.0, 0.5 / (gamma - 1.0)) * rho
    u, v = np.where(pick < 0.1, 0.0, u), np.where(pick < 0.1, 0.0, v)
    e = np.where((pick > 0.08) & (pick < 0.14), 0.0, e)
    energy = e + 0.5 * rho * (u * u + v * v)
    energy = np.where((pick > 0.13) & (pick < 0.15), -energy, energy)
    mx, my = rho * u, rho * v
    rho = np.where((pick > 0.2) & (pick < 0.22), 0.0, rho)
    a = np.stack((rho, energy, mx, my), axis=-1)
    _check(p, a, tile, f"{floors} thin {thin} gamma {gamma} riemann {riemann} tile {tile}")


@pytest.mark.parametrize("units", [3.49, 100.499])
@pytest.mark.parametrize("gamma", [1 + 2.0**-20, 1.4])
def test_largest_rate_at_the_lowest_floor(gpu_available, gamma, units):
    """Rates of energies that FP32 would keep in part, as in test_gpu_rate, at the lowest
    floor."""
    floor = 2.0**-110
    p = R._params(smallr=floor, smallc=floor, gamma0=gamma)
    lower = 0.5 * (units + np.floor(units)) / units
    e = units * 2.0**-149
    a = R._uniform(p, (floor / lower, e, 0.0), (floor, e, 0.0))
    R._compare(p, a, f"{units} units gamma {gamma}")
