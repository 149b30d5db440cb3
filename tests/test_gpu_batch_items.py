"""The items of the one-launch-per-step batch (balanced segments, shorter ones on
the edge strips, longest first) against the persistent launch, whose segments are
uniform: the same cells, so the same bits, at every tile.

Sizes: one, two and three strips, a last strip of one to four columns, fewer rows
than a tile, rows that no tile divides; and a batch whose wavefronts are resident
at once, two per SIMD, where they lower their issue priority as they go.
"""
import numpy as np
import pytest

from euler2d_kokkos_amd import (E2D_BATCH_LAUNCH_PERSISTENT, E2D_BATCH_LAUNCH_STEPS, E2D_LAYOUT_LEFT,
                                E2D_PRECISION_FP32_SPLIT, E2D_PRECISION_FP64)
from euler2d_kokkos_amd.batch import HydroBatch, make_params

pytestmark = pytest.mark.gpu

SHAPES = [(5, 4), (60, 7), (61, 64), (64, 65), (120, 27), (124, 33), (181, 5), (250, 131)]


def _params(shapes, slope):
    return [make_params(nx=nx, ny=ny, problemType=k % 2, gamma0=1.4, cfl=0.8, slope_type=slope,
                        nStepmax=1000, tEnd=1e9, honor_riemann=1, riemannSolverType=2,
                        implode_pressure_in=1.5, blast_radius=0.2, blast_center_x=0.5,
                        blast_center_y=0.5, blast_density_in=1.0, blast_density_out=1.0,
                        blast_pressure_in=10.0, blast_pressure_out=0.1,
                        boundary_type_xmin=1 + k % 3, boundary_type_xmax=1 + k % 3,
                        boundary_type_ymin=1, boundary_type_ymax=2)
            for k, (nx, ny) in enumerate(shapes)]


def _run(params, precision, mode, tile, steps):
    b = HydroBatch(params, precision=precision)
    b.set_launch(mode)
    b.set_tile(tile)
    b.run(steps)
    out = [(b.status(i), b.state(i, E2D_LAYOUT_LEFT)) for i in range(len(params))]
    b.close()
    return out


def _same(a, b):
    for k, ((sa, xa), (sb, xb)) in enumerate(zip(a, b)):
        assert sa == sb, k
        np.testing.assert_array_equal(xa, xb, err_msg=str(k))


@pytest.mark.parametrize("precision", [E2D_PRECISION_FP64, E2D_PRECISION_FP32_SPLIT])
@pytest.mark.parametrize("slope", [1.0, 2.0])
def test_items_cover_every_cell_once(gpu_available, precision, slope):
    params = _params(SHAPES, slope)
    ref = _run(params, precision, E2D_BATCH_LAUNCH_PERSISTENT, 16, 12)
    for tile in (1, 2, 5, 13, 27, 64, 4096):
        _same(_run(params, precision, E2D_BATCH_LAUNCH_STEPS, tile, 12), ref)


@pytest.mark.parametrize("precision", [E2D_PRECISION_FP64, E2D_PRECISION_FP32_SPLIT])
def test_items_resident_two_per_simd(gpu_available, precision):
    params = _params([(512, 512)] * 6 + [(384, 300)] * 2, 1.0)  # 20 rows: about 1600 wavefronts
    _same(_run(params, precision, E2D_BATCH_LAUNCH_STEPS, 20, 30),
          _run(params, precision, E2D_BATCH_LAUNCH_PERSISTENT, 20, 30))
