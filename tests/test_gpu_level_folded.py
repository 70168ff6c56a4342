"""The level tensor of an unshifted level, kept folded, against the same tensor built in full: every lane
grouping of its contraction (16, 32 and 64 layers, and one past each), lengths of the register and of the
LDS transforms, and a single row of blocks.

Tolerance: both sides take the same sums, up to a few thousand terms, in another order (segments, transforms,
layers): 2000 eps = 5e-13, times the cancellation between the four edges of a cell (below 100): 5e-11 of the
largest value, for the tensor's components and the field alike."""
import numpy as np
import pytest

from extreme_amd import cartesian_model as cm
from extreme_amd import xtreme as X

pytestmark = pytest.mark.gpu

TOL = 5e-11


@pytest.mark.parametrize("shape", [(6, 4, 3), (5, 12, 16), (8, 5, 17), (32, 6, 32), (4, 64, 33), (2, 2, 65)])
@pytest.mark.parametrize("electric", [True, False])
def test_folded_level_matches_full(torch_cuda, monkeypatch, shape, electric):
    torch = torch_cuda
    m = cm.small_model(*shape, seed=sum(shape))
    w = cm.omega_of(m.frequencies[0])
    rng = np.random.default_rng(shape[2])
    jq = torch.from_numpy(rng.standard_normal(m.n) + 1j * rng.standard_normal(m.n)).to("cuda")
    got = []
    for layout in ("full", None):
        monkeypatch.setenv("XTR_GREEN_LAYOUT", layout) if layout else monkeypatch.delenv("XTR_GREEN_LAYOUT")
        op = X.ConvolutionOperator(m, w)
        op.calculate_green_atoo(0.0, electric)
        field = op.level_field(jq, electric).cpu().numpy()
        op.calculate_green_atoo(0.0, electric, x_shift=m.dx)          # a shifted level in the same buffer, and back
        op.calculate_green_atoo(0.0, electric)
        again = op.level_field(jq, electric).cpu().numpy()
        assert np.array_equal(field, again)
        got.append((field, op.green_atoo(electric)))
    (f0, g0), (f1, g1) = got
    scale = max(np.abs(v).max() for v in g0.values())
    worst = max(np.abs(g1[c] - g0[c]).max() / scale for c in g0)
    err = np.abs(f1 - f0).max() / np.abs(f0).max()
    print(f"{shape} {'E' if electric else 'H'}: tensor {worst:.1e} field {err:.1e}", flush=True)
    assert set(g0) == set(g1) and worst < TOL and err < TOL
