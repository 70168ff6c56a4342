"""The folded contraction of blocks too large for LDS (a wave per 16 rows) against the generic per-wavenumber kernel:
depths on both sides of a full row tile and of a full k-step, of each swizzle of the tensor, and the largest.

Tolerances: a result sums 3 nz <= 255 products, so two orders of summation differ by at most about 255 eps of the sum
of magnitudes, a few times that of the result for random data: 1e-13 (complex128) and, with the transforms in
float32 as well, 2e-6 (complex64)."""
import numpy as np
import pytest

from tests.conftest import rel
from tests.test_gpu_block_contraction import _op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol,depths", [("fp64", 1e-13, (48, 49, 53, 56, 63, 65, 80, 85)),
                                                  ("fp32", 2e-6, (65, 72, 80, 85))])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 5])
def test_large_blocks_match_generic(oracle, torch_cuda, monkeypatch, nrhs, precision, tol, depths):
    torch = torch_cuda
    for nz in depths:
        if 3 * nz * nrhs > 1024:
            continue
        m, _, _, op = _op(oracle, (5, 4, nz), nrhs, precision, nz + nrhs)
        rng = np.random.default_rng(nz)
        x = torch.from_numpy(rng.standard_normal((nrhs, m.n)) + 1j * rng.standard_normal((nrhs, m.n))).to("cuda")
        y = op.apply(x).cpu().numpy()
        monkeypatch.setenv("XTR_CONTRACT_KERNEL", "generic")
        g = op.apply(x).cpu().numpy()
        monkeypatch.delenv("XTR_CONTRACT_KERNEL")
        e = max(rel(y[r], g[r]) for r in range(nrhs))
        print(f"nz {nz} nrhs {nrhs} {precision}: {e:.2e}", flush=True)
        assert e < tol, (nz, e)
