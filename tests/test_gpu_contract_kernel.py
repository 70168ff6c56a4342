"""Which contraction kernel an apply launches (xtr_op_contract_kernel, what the benchmark reports), and each of them
against the generic per-wavenumber kernel and the oracle on either side of the lines where another one takes over.

Tolerances: a result sums 3 nz <= 258 products, so two orders of summation differ by at most about 258 eps of the sum
of magnitudes, a few times that of the result for random data: 1e-13 (complex128), and 1e-12 against the oracle, whose
transforms differ too; with the transforms in float32 as well 2e-6 (complex64)."""
import numpy as np
import pytest

from tests.conftest import rel
from tests.test_gpu_block_contraction import _op

pytestmark = pytest.mark.gpu


def _x(m, nrhs, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal((nrhs, m.n)) + 1j * rng.standard_normal((nrhs, m.n))


# a wave per block from 6 blocks a CU (2 up to 5 layers) on; (24, 20), (20, 20): 525 and 441 blocks; (40, 40), (40, 32): 1681, 1353
@pytest.mark.parametrize("grid,nz,nrhs,direct", [((24, 20), 5, 2, True), ((20, 20), 5, 2, False), ((24, 20), 3, 8, True),
                                                 ((20, 20), 3, 8, False), ((40, 40), 8, 2, True), ((40, 32), 8, 2, False),
                                                 ((40, 40), 10, 5, True), ((40, 32), 10, 5, False), ((40, 40), 11, 2, False)])
@pytest.mark.parametrize("precision,tol_g,tol_o", [("fp64", 1e-13, 1e-12), ("fp32", 2e-6, 2e-6)])
def test_few_layers_on_either_side(oracle, torch_cuda, monkeypatch, grid, nz, nrhs, direct, precision, tol_g, tol_o):
    if torch_cuda.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the grids lie on either side of the line of a chip with 256 CUs")
    m, w, G, op = _op(oracle, (*grid, nz), nrhs, precision, nz + nrhs)
    assert op.contract_kernel(nrhs) is None
    xs = _x(m, nrhs, nz)
    y = op.apply(xs)
    kernel = op.contract_kernel(nrhs)
    assert kernel.startswith(f"contract_{'direct' if direct else 'block'}_kernel<{'double' if precision == 'fp64' else 'float'}, {nz}, ")
    monkeypatch.setenv("XTR_CONTRACT_KERNEL", "generic")
    g = op.apply(xs)
    assert op.contract_kernel(nrhs) == f"contract_kernel<{'double' if precision == 'fp64' else 'float'}>"
    oop = oracle.Operator(m, G)
    oop.prepare("A", m.zeta(w).reshape(-1), m.zeta0(w))
    eg = max(rel(y[r], g[r]) for r in range(nrhs))
    eo = max(rel(y[r], oop.apply(xs[r])) for r in {0, nrhs - 1})
    print(f"{grid} nz {nz} nrhs {nrhs} {kernel}: vs generic {eg:.1e}, vs oracle {eo:.1e}", flush=True)
    assert eg < tol_g and eo < tol_o


@pytest.mark.parametrize("nz,nrhs,precision,layout,kernel", [
    (32, 2, "fp64", None, "contract_block_kernel<double, 32, 2>"), (47, 1, "fp64", None, "contract_block_kernel<double, 47, 1>"),
    (24, 3, "fp64", None, "contract_block_kernel<double, 24, 2>"), (48, 2, "fp64", None, "contract_rows_kernel<double, 1>"),
    (48, 2, "fp32", None, "contract_block_kernel<float, 48, 2>"), (85, 3, "fp64", None, "contract_rows_kernel<double, 2>"),
    (86, 2, "fp64", None, "contract_kernel<double>"), (64, 2, "fp64", None, "contract_fold64_kernel<double>"),
    (64, 3, "fp32", None, "contract_fold64_kernel<float>"), (32, 2, "fp64", "full", "contract_stream_kernel<double>"),
    (64, 2, "fp64", "full", "contract_stream64_kernel<double, 2>"), (24, 2, "fp64", "full", "contract_kernel<double>")])
def test_kernel_by_depth_and_layout(oracle, torch_cuda, monkeypatch, nz, nrhs, precision, layout, kernel):
    if layout:
        monkeypatch.setenv("XTR_GREEN_LAYOUT", layout)
    from extreme_amd import cartesian_model as cm
    from extreme_amd import xtreme as X
    m = cm.small_model(4, 5, nz, seed=nz)
    op = X.ConvolutionOperator(m, cm.omega_of(m.frequencies[0]), precision=precision, max_rhs=nrhs)
    op.calculate_green_tensor()
    op.prepare_operator("A")
    op.apply(_x(m, nrhs, nz))
    assert op.contract_kernel(nrhs) == kernel
    if nrhs > 1:
        assert op.contract_kernel(1) is None
    with pytest.raises(X.XtrError, match="nrhs"):
        op.contract_kernel(nrhs + 1)
