"""Host copies of the state through the staging kernels.

Sizes: one partial tile, a few tiles, several chunks through one thread's two
buffers, and enough for the copying threads; every layout and precision, against
numpy's own reordering of one upload.
"""
import numpy as np
import pytest

from euler2d_kokkos_amd import (E2D_LAYOUT_INTERIOR, E2D_LAYOUT_LEFT, E2D_LAYOUT_RIGHT,
                                E2D_PRECISION_FP32, E2D_PRECISION_FP32_SPLIT, E2D_PRECISION_FP64,
                                E2D_U, E2D_U2, HydroParams, HydroRun)
from euler2d_kokkos_amd.batch import make_params

pytestmark = pytest.mark.gpu

PRECISIONS = {"fp64": E2D_PRECISION_FP64, "split": E2D_PRECISION_FP32_SPLIT,
              "fp32": E2D_PRECISION_FP32}


def _stored(x, precision):
    """What the device keeps of FP64 values."""
    hi = x.astype(np.float32)
    if precision == E2D_PRECISION_FP64:
        return x
    if precision == E2D_PRECISION_FP32:
        return hi.astype(np.float64)
    return hi.astype(np.float64) + (x - hi.astype(np.float64)).astype(np.float32)


@pytest.mark.parametrize("precision", sorted(PRECISIONS))
@pytest.mark.parametrize("nx,ny", [(2, 3), (61, 67), (13, 9000), (700, 530), (1100, 801)])
def test_state_copies(gpu_available, nx, ny, precision):
    prec = PRECISIONS[precision]
    p = HydroParams(make_params(nx=nx, ny=ny, problemType=1))
    run = HydroRun(p, precision=prec, initialise=False)
    rng = np.random.default_rng(nx)
    planes = rng.standard_normal((4, ny + 4, nx + 4)) * 10.0 ** rng.integers(-3, 4, (4, 1, 1))
    kept = _stored(planes, prec)
    run.set_state(E2D_U, planes, E2D_LAYOUT_LEFT)
    run.set_state(E2D_U2, np.ascontiguousarray(planes.transpose(2, 1, 0)), E2D_LAYOUT_RIGHT)
    for which in (E2D_U, E2D_U2):
        np.testing.assert_array_equal(run.get_state(which, E2D_LAYOUT_LEFT), kept)
        np.testing.assert_array_equal(run.get_state(which, E2D_LAYOUT_RIGHT),
                                      kept.transpose(2, 1, 0))
        np.testing.assert_array_equal(run.get_state(which, E2D_LAYOUT_INTERIOR),
                                      kept[:, 2:-2, 2:-2])
    # an interior upload leaves the ghost cells alone
    inner = rng.standard_normal((4, ny, nx))
    run.set_state(E2D_U, inner, E2D_LAYOUT_INTERIOR)
    want = kept.copy()
    want[:, 2:-2, 2:-2] = _stored(inner, prec)
    np.testing.assert_array_equal(run.get_state(E2D_U, E2D_LAYOUT_LEFT), want)
    np.testing.assert_array_equal(run.get_state(E2D_U2, E2D_LAYOUT_LEFT), kept)
