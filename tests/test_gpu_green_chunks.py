"""Assembly of an anomaly tensor whose layer pairs pass in several chunks, the last one no multiple of 8: 50 layers have
1275 symmetric pairs (284 MB of U, chunks of 640 and 635) and 2500 others (186 MB, 1256 and 1244), in two background
layers, against the oracle.

Tolerance: the kernels take the oracle's sums in another order; up to 2000 terms and a cancellation between a cell's
edges below 100 give 2000 x 100 x eps = 5e-11 of a component's largest value. A pair taken for another one differs by its own
size: the smallest pair's largest value is 7e-8 of its component's."""
import numpy as np
import pytest

from extreme_amd import cartesian_model as cm
from extreme_amd import xtreme as X

pytestmark = pytest.mark.gpu

TOL = 5e-11


def _model():
    thick = np.array([100.0] * 20 + [200.0] * 30)
    depth = np.concatenate([[0.0], np.cumsum(thick)[:-1]])
    sec = cm.Section1D(0.0, [0.0, 2000.0, 8000.0, 0.0], [0.0, 1e-2, 1e-1, 1e-3])
    return cm.CartesianModel(3, 2, 200.0, 250.0, depth, thick, np.full((3, 2, 50), 0.05), sec, "chunks", [0.3])


@pytest.mark.parametrize("layout", [None, "full"])
def test_pairs_in_several_chunks(oracle, torch_cuda, monkeypatch, layout):
    if layout:
        monkeypatch.setenv("XTR_GREEN_LAYOUT", layout)
    m = _model()
    w = cm.omega_of(m.frequencies[0])
    op = X.ConvolutionOperator(m, w)
    op.calculate_green_tensor()
    got, ref = op.green_tensor(), oracle.green_atoa(m, w)
    for c in ref:
        e = np.abs(got[c] - ref[c]).max(axis=0) / np.abs(ref[c]).max()
        print(f"{layout or 'folded'} {c}: {e.max():.1e} at pair {e.argmax()}", flush=True)
        assert e.max() < TOL, c
