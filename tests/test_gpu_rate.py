"""The largest CFL rate of a step, whatever the tile.

The time step follows from the largest rate of the step's output, which its wavefronts
fold as they march; tiles of eight rows and of seven are different kernels (two rows
loaded ahead, or one), and at these sizes eight rows are more than two rounds of
wavefronts.  The times and the arrays of the two must agree bit for bit, also where the
largest rate belongs to a few cells that a shorter or narrower evaluation would miss:
the grid's lower part holds states of slightly smaller rate, in the wavefronts that
march first, and its upper part the cell state in question.
"""
import numpy as np
import pytest

import oracle_lib as O
from euler2d_kokkos_amd import E2D_U, E2D_U2, HydroParams, HydroRun, device_info

pytestmark = pytest.mark.gpu

NX, NY, STEPS = 1024, 2048, 3
CUT = 1700  # first row of the upper part


def _params(nx=NX, ny=NY, **more):
    f = dict(nx=nx, ny=ny, ymax=ny / nx, cfl=0.5, nStepmax=STEPS, tEnd=1e300, problemType=1,
             honor_riemann=1, riemannSolverType=2, boundary_type_xmin=3, boundary_type_xmax=3,
             boundary_type_ymin=2, boundary_type_ymax=2)
    f.update(more)
    return O.default_params(**f)


def _run(p, tile, a):
    strips = (p.nx + 59) // 60
    if tile == 8:  # more than two rounds of two wavefronts per SIMD
        assert strips * ((p.ny + 7) // 8) > 4 * 4 * device_info()[1]
    run = HydroRun(HydroParams(p.copy()), initialise=False)
    run.set_tile(tile)
    for which in (E2D_U, E2D_U2):
        run.set_state(which, a)
    run.run()
    out = run.t, run.nStep, run.get_state(E2D_U), run.get_state(E2D_U2)
    run.close()
    return out


def _compare(p, a, what):
    t8, n8, u8, v8 = _run(p, 8, a)
    t7, n7, u7, v7 = _run(p, 7, a)
    assert n8 == n7 == STEPS, what
    assert t8 == t7, what
    for g, o in ((u8, u7), (v8, v7)):
        assert np.array_equal(g.view(np.int64), o.view(np.int64)), what


def _uniform(p, lower, upper):
    """(rho, pressure / (gamma - 1), x velocity) below row CUT and from it on."""
    a = np.zeros((p.isize, p.jsize, 4))
    for rows, (rho, e, u) in ((slice(None, CUT), lower), (slice(CUT, None), upper)):
        a[:, rows, 0] = rho
        a[:, rows, 1] = e + 0.5 * rho * u * u
        a[:, rows, 2] = rho * u
    return a


# (lower part, upper part): the upper part's rate is the larger one.  The contact
# between them is at rest across, and its pressures are equal where the values
# allow it, so the states stay as they are.
FLOOR = 2.0**-60
STATES = {
    # speeds whose square is outside FP32, energies inside and outside it
    "fast": ((0.263, 1e38, 0.0), (1.0, 1e38, 2e19)),
    "fast and hot": ((2.6e21, 1e60, 0.0), (1.0, 1e60, 2e19)),
    # energies below FP32's range at the density floor
    "cold": ((0.56 * 2.0**-41, 2.0**-151, 0.0), (FLOOR, 2.0**-151, 0.0)),
    # in range
    "ordinary": ((1.0, 2.5, 0.3), (1.0, 2.5, 0.4)),
    "supersonic": ((1.0, 2.5, 0.0), (1.0, 2.5, 1e6)),
}


@pytest.mark.parametrize("riemann", [1, 2], ids=["hll", "hllc"])
@pytest.mark.parametrize("state", sorted(STATES))
def test_largest_rate_is_kept(gpu_available, state, riemann):
    floors = dict(smallr=FLOOR, smallc=FLOOR) if state == "cold" else {}
    p = _params(riemannSolverType=riemann, **floors)
    _compare(p, _uniform(p, *STATES[state]), f"{state} riemann {riemann}")


@pytest.mark.parametrize("slope", [1.0, 2.0], ids=["minmod", "mc"])
@pytest.mark.parametrize("nx", [1000, 1024])
def test_largest_rate_of_a_field(gpu_available, nx, slope):
    """Random cells, among them ones of far higher speed, of vanishing pressure
    beside their kinetic energy, and at the floors."""
    p = _params(nx=nx, ny=2200, slope_type=slope, riemannSolverType=1 + nx % 3 % 2)
    rng = np.random.default_rng(11)
    shape = (p.isize, p.jsize)
    rho, u, v = np.exp(rng.normal(0, 1, shape)), rng.normal(0, 1, shape), rng.normal(0, 1, shape)
    e = np.exp(rng.normal(0, 1, shape))
    pick = rng.random(shape)
    u = np.where(pick < 0.002, 40.0 * u, u)
    e = np.where((pick > 0.1) & (pick < 0.15), 1e-13, e)
    rho = np.where((pick > 0.2) & (pick < 0.21), p.smallr, rho)
    a = np.stack((rho, e * rho + 0.5 * rho * (u * u + v * v), rho * u, rho * v), axis=-1)
    _compare(p, a, f"field {nx} slope {slope}")


@pytest.mark.parametrize("riemann", [1, 2], ids=["hll", "hllc"])
@pytest.mark.parametrize("units", [3.49, 8.499, 100.499])
def test_largest_rate_of_partly_lost_energies(gpu_available, units, riemann):
    """Energies of a few units of FP32's smallest number, which FP32 would round down, at
    the density floor.  The lower part has the same pressure, and a density that puts
    its rate between the upper part's and the one that the rounded energy would give."""
    p = _params(riemannSolverType=riemann, smallr=FLOOR, smallc=FLOOR)
    e = units * 2.0**-149
    lower = 0.5 * (units + np.floor(units)) / units  # its squared rate over the upper part's
    a = _uniform(p, (FLOOR / lower, e, 0.0), (FLOOR, e, 0.0))
    _compare(p, a, f"{units} units riemann {riemann}")
