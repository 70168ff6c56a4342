"""Green assembly where few pairs or few cells split the work differently: pairs in groups of 16 to 256 threads,
offsets near the receiver shared by a workgroup and the others by a wave (a shifted level moves that window off
the middle, to an edge and beyond), and radii shared by workgroups of the Hankel filter; against the oracle.

Tolerance: the kernels take the oracle's sums in another order; up to 2000 terms and a cancellation between a
cell's edges below 100 give 2000 x 100 x eps = 5e-11 of the largest value."""
import numpy as np
import pytest

from extreme_amd import cartesian_model as cm
from extreme_amd import xtreme as X

pytestmark = pytest.mark.gpu

TOL = 5e-11


def _close(got, ref, tag):
    scale = max(np.abs(v).max() for v in ref.values())
    worst = max(np.abs(got[c] - ref[c]).max() / scale for c in ref)
    print(f"{tag}: {worst:.1e}", flush=True)
    assert worst < TOL, tag


@pytest.mark.parametrize("shape", [(3, 2, 1), (5, 4, 5), (12, 6, 6), (4, 3, 11), (2, 2, 17)])
def test_anomaly_tensor_in_pair_groups(oracle, torch_cuda, shape):
    m = cm.small_model(*shape, seed=sum(shape))
    w = cm.omega_of(m.frequencies[0])
    op = X.ConvolutionOperator(m, w)
    op.calculate_green_tensor()
    ref = oracle.green_atoa(m, w)
    got = op.green_tensor()
    _close(got, ref, f"{shape}")


@pytest.mark.parametrize("shape,shift", [((24, 16, 3), (0.0, 0.0)), ((24, 16, 9), (11.0, -7.25)), ((16, 4, 2), (-14.5, 40.0)),
                                         ((3, 20, 17), (0.4, 19.0))])
@pytest.mark.parametrize("electric", [True, False])
def test_level_tensor_near_and_far(oracle, torch_cuda, shape, shift, electric):
    m = cm.small_model(*shape, seed=sum(shape))
    w = cm.omega_of(m.frequencies[0])
    sx, sy = shift[0] * m.dx, shift[1] * m.dy
    op = X.ConvolutionOperator(m, w)
    op.calculate_green_atoo(0.0, electric, x_shift=sx, y_shift=sy)
    _close(op.green_atoo(electric), oracle.green_atoo_level(m, w, 0.0, electric, x_shift=sx, y_shift=sy),
           f"{shape} {shift} {'E' if electric else 'H'}")


@pytest.mark.parametrize("shape", [(32, 32, 12), (4, 256, 12), (64, 20, 17)])
def test_cells_near_the_source_apart_from_the_others(oracle, torch_cuda, shape):
    """Enough cells and pairs that the cells within 8 of the source take a launch of their own."""
    m = cm.small_model(*shape, seed=sum(shape))
    w = cm.omega_of(m.frequencies[0])
    op = X.ConvolutionOperator(m, w)
    op.calculate_green_tensor()
    ref = oracle.green_atoa(m, w)
    _close(op.green_tensor(), ref, f"{shape}")
