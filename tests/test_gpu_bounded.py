"""The bounded FP64 step kinds at the edges of their ranges.

The fused FP64 step forms its quotients without scaling steps where every cell a
wavefront reads is in checked ranges (density, pressure, velocity, magnitude of
small numerators, dt / dx), and takes the reference's operations elsewhere.  A
few cells on either side of each edge, scattered over a smooth state, make
wavefronts go from one path to the other and back within a march; every array
must equal the CPU oracle's bit for bit, the sign of zeros included.
"""
import numpy as np
import pytest

import oracle_lib as O
from euler2d_kokkos_amd import E2D_U, E2D_U2, HydroParams, HydroRun

pytestmark = pytest.mark.gpu

BASE = dict(nx=130, ny=45, cfl=0.5, nStepmax=5, tEnd=1e9, problemType=1, blast_radius=0.3,
            honor_riemann=1)
# value lists straddle an edge: density 2^40, pressure 2^90, velocity ~2^50,
# numerators 2^-969, signed zeros
EDGES = {
    "density": ("rho", [2.0**40, 2.0**40 * (1 + 2.0**-52), 2.0**41, 1e20]),
    "pressure": ("energy", [2.0**91, 3.2e27, 1e29]),
    "velocity": ("mom", [2.0**50, -2.0**50, 2.0**51, 1.2e15]),
    "tiny": ("mom", [0.0, -0.0, 2.0**-968, -2.0**-970, 1e-300, -5e-324, 5e-324, 1e-310]),
    "rest": ("mom", [0.0, -0.0]),
}


def _state(p, edge, seed):
    ora = O.OracleRun(p)
    a = ora.get(0)
    rng = np.random.default_rng(seed)
    x = np.arange(a.shape[0])[:, None] / 20.0
    y = np.arange(a.shape[1])[None, :] / 9.0
    rho = 1.0 + 0.3 * np.sin(x) * np.cos(y)
    u, v, pr = 0.4 * np.cos(x + y), -0.3 * np.sin(y), 1.0 + 0.2 * np.cos(x)
    if edge == "rest":
        u, v = np.zeros_like(rho), np.zeros_like(rho)
    kind, vals = EDGES[edge]
    mask = rng.random(rho.shape) < (0.02 if edge in ("density", "pressure", "velocity") else 0.2)
    pick = np.asarray(vals)[rng.integers(0, len(vals), size=rho.shape)]
    if kind == "rho":
        rho = np.where(mask, pick, rho)
    mx, my = rho * u, rho * v
    if kind == "mom":
        mx, my = np.where(mask, pick, mx), np.where(np.roll(mask, 3), pick, my)
    e = pr / (p.gamma0 - 1.0) + 0.5 * (mx * mx + my * my) / rho
    if kind == "energy":
        e = np.where(mask, pick, e)
    a[..., 0], a[..., 1], a[..., 2], a[..., 3] = rho, e, mx, my
    return ora, a


def _same_bits(run, ora, what):
    assert (run.t, run.nStep) == (ora.t, ora.nStep), what
    for which in (E2D_U, E2D_U2):
        g, o = run.get_state(which), ora.get(which)
        # velocities of 2^50 and more absorb the sound speed: HLLC's own quotients
        # turn NaN there, in the oracle as well
        nan = np.isnan(o)
        np.testing.assert_array_equal(np.isnan(g), nan, err_msg=what)
        np.testing.assert_array_equal(g.view(np.int64)[~nan], o.view(np.int64)[~nan],
                                      err_msg=what)


@pytest.mark.parametrize("tile", [1, 7, 16])
@pytest.mark.parametrize("riemann", [1, 2], ids=["hll", "hllc"])
@pytest.mark.parametrize("slope", [1.0, 2.0], ids=["minmod", "mc"])
@pytest.mark.parametrize("edge", sorted(EDGES))
def test_bounded_kinds_at_their_edges(gpu_available, edge, slope, riemann, tile):
    # 128 columns: power-of-two cells, the deck kernels; 130: the general ones
    p = O.default_params(**dict(BASE, nx=128 if slope == 1.0 else 130, riemannSolverType=riemann,
                                slope_type=slope))
    ora, a = _state(p, edge, seed=7)
    for which in (0, 1):
        ora.set(which, a)
    run = HydroRun(HydroParams(p.copy()))
    run.set_tile(tile)
    run.set_state(E2D_U, a)
    run.set_state(E2D_U2, a)
    ora.run()
    run.run()
    _same_bits(run, ora, f"{edge} slope {slope} riemann {riemann} tile {tile}")


def test_bounded_kinds_long_time_step(gpu_available):
    """A cold gas at rest (pressure floor, smallc 1e-15): dt / dx is above 2^40,
    so every wavefront takes the reference's operations."""
    p = O.default_params(**dict(BASE, smallc=1e-15, riemannSolverType=2))
    ora, a = _state(p, "rest", seed=3)
    a[..., 1] = 0.0
    for which in (0, 1):
        ora.set(which, a)
    run = HydroRun(HydroParams(p.copy()))
    run.set_state(E2D_U, a)
    run.set_state(E2D_U2, a)
    assert run.compute_dt(0) * p.nx > 2.0**40
    ora.run()
    run.run()
    _same_bits(run, ora, "cold gas")
