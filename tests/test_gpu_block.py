"""The block step kernel at the edges of its blocks.

Tiles of up to 20 rows whose blocks fit one per CU run the block kernel: one
loaded row per wavefront up to 12 rows, two above.  Grids narrower and wider than
one strip of 60 columns, shorter than a block, exactly one, and one row more;
FP64 against the CPU oracle, split precision against the march (a tile above 20
rows), bit for bit, ghost cells included.
"""
import numpy as np
import pytest

import oracle_lib as O
from euler2d_kokkos_amd import (E2D_PRECISION_FP32_SPLIT, E2D_PRECISION_FP64, E2D_U, E2D_U2,
                                HydroParams, HydroRun)

pytestmark = pytest.mark.gpu

GRIDS = [(2, 2), (3, 41), (59, 12), (60, 13), (61, 20), (121, 21), (180, 39)]


def _params(nx, ny, **more):
    bc = {1: (1, 1, 1, 1), 2: (2, 2, 3, 3), 0: (3, 3, 1, 2)}[(nx + ny) % 3]
    f = dict(nx=nx, ny=ny, problemType=1, blast_radius=0.25, cfl=0.7, nStepmax=7, tEnd=1e9,
             ymax=ny / nx, boundary_type_xmin=bc[0], boundary_type_xmax=bc[1],
             boundary_type_ymin=bc[2], boundary_type_ymax=bc[3], honor_riemann=1)
    f.update(more)
    return O.default_params(**f)


def _run(p, tile, precision=E2D_PRECISION_FP64):
    run = HydroRun(HydroParams(p.copy()), precision=precision)
    run.set_tile(tile)
    run.run(3)
    run.run()
    return run


@pytest.mark.parametrize("tile", [1, 2, 11, 12, 13, 20])
@pytest.mark.parametrize("nx,ny", GRIDS)
def test_block_matches_oracle(gpu_available, nx, ny, tile):
    riemann = 1 + (nx + tile) % 2
    p = _params(nx, ny, riemannSolverType=riemann, slope_type=float(1 + tile % 2))
    ora = O.OracleRun(p)
    ora.run()
    run = _run(p, tile)
    assert (run.t, run.nStep) == (ora.t, ora.nStep)
    for which in (E2D_U, E2D_U2):
        np.testing.assert_array_equal(run.get_state(which).view(np.int64),
                                      ora.get(which).view(np.int64))


@pytest.mark.parametrize("tile", [1, 7, 12, 14, 20])
@pytest.mark.parametrize("nx,ny", GRIDS)
def test_block_split_matches_march(gpu_available, nx, ny, tile):
    p = _params(nx, ny, riemannSolverType=1 + (ny + tile) % 2, kin_frac=0.3)
    a = _run(p, tile, E2D_PRECISION_FP32_SPLIT)
    b = _run(p, 24, E2D_PRECISION_FP32_SPLIT)
    assert (a.t, a.nStep) == (b.t, b.nStep)
    for which in (E2D_U, E2D_U2):
        np.testing.assert_array_equal(a.get_state(which), b.get_state(which))


def test_block_step_with_given_dt(gpu_available):
    """godunov_unsplit (no loop state) on the block kernel against the march."""
    p = _params(130, 37, riemannSolverType=2)
    runs = []
    for tile in (5, 18, 30):
        r = HydroRun(HydroParams(p.copy()))
        r.set_tile(tile)
        for n in range(5):
            r.godunov_unsplit(n, 0.5 * r.compute_dt(n % 2))
        runs.append([r.get_state(w) for w in (E2D_U, E2D_U2)])
    for got in runs[:2]:
        for g, want in zip(got, runs[2]):
            np.testing.assert_array_equal(g, want)
