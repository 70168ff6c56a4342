"""The folded contraction with a wave per block (few layers, many blocks): every depth it takes against the generic
per-wavenumber kernel, at grids just past where it starts, with edge blocks and a last, partly filled workgroup.

Tolerances: a result sums 3 nz <= 30 products, so two orders of summation differ by at most about 30 eps of the sum
of magnitudes, a few times that of the result for random data: 1e-13 (complex128) and, with the transforms in
float32 as well, 2e-6 (complex64)."""
import numpy as np
import pytest

from tests.conftest import rel
from tests.test_gpu_block_contraction import _op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-13), ("fp32", 2e-6)])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("grid,depths", [((20, 24), (1, 2, 3, 4, 5)), ((40, 40), (5, 6, 7, 8, 9, 10))])
def test_every_depth_matches_generic(oracle, torch_cuda, monkeypatch, grid, depths, nrhs, precision, tol):
    torch = torch_cuda
    worst = (0.0, 0)
    for nz in depths:
        m, _, _, op = _op(oracle, (*grid, nz), nrhs, precision, nz + nrhs)
        rng = np.random.default_rng(nz)
        x = torch.from_numpy(rng.standard_normal((nrhs, m.n)) + 1j * rng.standard_normal((nrhs, m.n))).to("cuda")
        y = op.apply(x).cpu().numpy()
        monkeypatch.setenv("XTR_CONTRACT_KERNEL", "generic")
        g = op.apply(x).cpu().numpy()
        monkeypatch.delenv("XTR_CONTRACT_KERNEL")
        e = max(rel(y[r], g[r]) for r in range(nrhs))
        worst = max(worst, (e, nz))
        assert e < tol, (nz, e)
    print(f"{grid} nrhs {nrhs} {precision}: worst {worst[0]:.2e} at nz = {worst[1]}", flush=True)
