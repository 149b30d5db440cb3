"""The bounded FP64 quotients on the march.

Small grids at tiles of up to 20 rows run the block kernel; every larger grid and
every batch marches, with its own way of carrying a row's checks to the rows after
it and of redoing a row with the reference's operations.  Here the march gets the
states at the edges of the ranges: tiles above 20 rows, tiles of three rows on a
grid of more blocks than the block kernel takes (one row loaded ahead), and batches
in both launches.  Every array must equal the CPU oracle's bit for bit.
"""
import numpy as np
import pytest

import oracle_lib as O
from euler2d_kokkos_amd import (E2D_BATCH_LAUNCH_PERSISTENT, E2D_BATCH_LAUNCH_STEPS,
                                E2D_PRECISION_FP64, E2D_U, E2D_U2, HydroParams, HydroRun,
                                device_info)
from euler2d_kokkos_amd.batch import HydroBatch
from test_gpu_bounded import BASE, EDGES, _same_bits, _state

pytestmark = pytest.mark.gpu


def _run(p, tile, a):
    blocks = ((p.nx + 59) // 60) * ((p.ny + tile - 1) // tile)
    assert tile > 20 or blocks > device_info()[1]  # else the block kernel takes it
    run = HydroRun(HydroParams(p.copy()))
    run.set_tile(tile)
    run.set_state(E2D_U, a)
    run.set_state(E2D_U2, a)
    run.run()
    return run


def _oracle(ora, a):
    for which in (0, 1):
        ora.set(which, a)
    ora.run()
    return ora


@pytest.mark.parametrize("tile", [3, 24, 45])
@pytest.mark.parametrize("riemann", [1, 2], ids=["hll", "hllc"])
@pytest.mark.parametrize("slope", [1.0, 2.0], ids=["minmod", "mc"])
@pytest.mark.parametrize("nx", [128, 130])  # power-of-two cells or not
@pytest.mark.parametrize("edge", sorted(EDGES))
def test_march_at_the_edges(gpu_available, edge, nx, slope, riemann, tile):
    wide = 8 if tile == 3 else 1  # 1024 or 1040 columns: 18 strips of 15 segments
    p = O.default_params(**dict(BASE, nx=nx * wide, ymax=45.0 / 128, riemannSolverType=riemann,
                                slope_type=slope))
    ora, a = _state(p, edge, seed=7)
    run = _run(p, tile, a)
    _same_bits(run, _oracle(ora, a), f"{edge} nx {nx} slope {slope} riemann {riemann} tile {tile}")


@pytest.mark.parametrize("tile", [24, 45])
def test_march_of_a_long_time_step(gpu_available, tile):
    """dt / dx above 2^40: every wavefront takes the reference's operations."""
    p = O.default_params(**dict(BASE, smallc=1e-15, riemannSolverType=2))
    ora, a = _state(p, "rest", seed=3)
    a[..., 1] = 0.0
    _same_bits(_run(p, tile, a), _oracle(ora, a), f"cold gas, tile {tile}")


@pytest.mark.parametrize("mode", [E2D_BATCH_LAUNCH_STEPS, E2D_BATCH_LAUNCH_PERSISTENT],
                         ids=["steps", "persistent"])
@pytest.mark.parametrize("riemann", [1, 2], ids=["hll", "hllc"])
@pytest.mark.parametrize("slope", [1.0, 2.0], ids=["minmod", "mc"])
def test_batch_past_the_edges(gpu_available, slope, riemann, mode):
    """Blasts whose disc is inside, at or past a bound of density or pressure, in one
    batch with an ordinary one."""
    inside = [(1.0, 10.0), (2.0**40, 10.0), (2.0**40 * (1 + 2.0**-52), 10.0), (1e20, 10.0),
              (1.0, 2.0**89.5), (1.0, 3.2e27), (1.0, 1e29), (1e26, 1e50)]
    raw = []
    for k, (rho, pr) in enumerate(inside):
        nx, ny = 64 + 33 * (k % 3), 50 + 17 * (k % 2)
        raw.append(O.default_params(
            nx=nx, ny=ny, ymax=ny / nx, cfl=0.6, nStepmax=12, tEnd=1e9, problemType=1,
            blast_radius=0.2, blast_center_x=0.5, blast_center_y=0.4, blast_density_in=rho,
            blast_density_out=1.0, blast_pressure_in=pr, blast_pressure_out=0.1,
            honor_riemann=1, riemannSolverType=riemann, slope_type=slope))
    for tile in (7, 30):
        b = HydroBatch([p.copy() for p in raw], precision=E2D_PRECISION_FP64)
        b.set_launch(mode)
        b.set_tile(tile)
        b.run(12)
        for i, p in enumerate(raw):
            ora = O.OracleRun(p)
            ora.run()
            what = f"instance {i} tile {tile}"
            assert b.status(i) == (ora.t, ora.nStep), what
            got, want = b.state(i), ora.get(ora.nStep % 2)
            nan = np.isnan(want)
            np.testing.assert_array_equal(np.isnan(got), nan, err_msg=what)
            np.testing.assert_array_equal(got.view(np.int64)[~nan], want.view(np.int64)[~nan],
                                          err_msg=what)
        b.close()
