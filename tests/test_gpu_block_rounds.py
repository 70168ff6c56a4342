"""The contraction with a block in LDS where workgroups of two and three waves (up to 16 layers) take several blocks:
from the second block on its waits count the stores of the one before and the copies of the next. A CU holds 32 waves,
so at most 10 workgroups of three waves (11 to 16 layers: 3900 blocks and more for 2560 workgroups). Up to 10 layers
the block kernel has fewer than 1536 blocks; eight right-hand sides in two groups of 4 leave a group 128 times the
workgroups of a CU, at most 8 of three waves and, in complex128, of two by registers (1353 blocks for 1024).

Tolerances: a result sums 3 nz <= 48 products, so two orders of summation differ by at most about 48 eps of the sum
of magnitudes, a few times that of the result for random data: 1e-13 (complex128) and, with the transforms in
float32 as well, 2e-6 (complex64)."""
import numpy as np
import pytest

from tests.conftest import rel
from tests.test_gpu_contract_kernel import _op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,counts", [((64, 60, 11), (1, 2, 3, 4)), ((60, 64, 13), (1, 2, 4, 8)), ((64, 64, 16), (1, 2, 3, 8)),
                                          ((40, 32, 10), (8,)), ((40, 32, 8), (8,))])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-13), ("fp32", 2e-6)])
def test_small_workgroups_take_several_blocks(oracle, torch_cuda, monkeypatch, shape, counts, precision, tol):
    m, _, _, op = _op(oracle, shape, max(counts), precision, sum(shape))
    rng = np.random.default_rng(shape[2])
    xs = rng.standard_normal((max(counts), m.n)) + 1j * rng.standard_normal((max(counts), m.n))
    for nrhs in counts:
        y = op.apply(xs[:nrhs])
        kernel = op.contract_kernel(nrhs)
        assert kernel.startswith("contract_block_kernel")
        monkeypatch.setenv("XTR_CONTRACT_KERNEL", "generic")
        g = op.apply(xs[:nrhs])
        monkeypatch.delenv("XTR_CONTRACT_KERNEL")
        e = max(rel(y[r], g[r]) for r in range(nrhs))
        print(f"{shape} nrhs {nrhs} {kernel}: {e:.2e}", flush=True)
        assert e < tol
