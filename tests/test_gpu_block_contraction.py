"""The folded contraction with a block in LDS (one kernel per depth): every depth against the generic
per-wavenumber kernel, and several blocks per workgroup against the oracle.

Tolerances: a result sums 3 nz <= 192 products, so two orders of summation differ by at most about
192 eps of the sum of magnitudes, a few times that of the result for random data: 1e-13 (complex128)
and, with the transforms in float32 as well, 2e-6 (complex64)."""
import numpy as np
import pytest

from extreme_amd import cartesian_model as cm
from extreme_amd import xtreme as X
from tests.conftest import rel
from tests.test_gpu_folded import _mirror_symmetric_green

pytestmark = pytest.mark.gpu


def _op(oracle, shape, nrhs, precision, seed):
    m = cm.small_model(*shape, seed=seed)
    w = cm.omega_of(m.frequencies[0])
    G = _mirror_symmetric_green(oracle, m, seed)
    op = X.ConvolutionOperator(m, w, precision=precision, max_rhs=nrhs)
    op.set_green_tensor(G)
    assert op.green_layout()[0] == "folded"
    op.prepare_operator("A")
    return m, w, G, op


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-13), ("fp32", 2e-6)])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 5, 8])
def test_every_depth_matches_generic(oracle, torch_cuda, monkeypatch, nrhs, precision, tol):
    torch = torch_cuda
    worst = (0.0, 0)
    for nz in range(1, 65):
        if 3 * nz * nrhs > 1024:
            continue
        m, _, _, op = _op(oracle, (4, 5, nz), nrhs, precision, nz + nrhs)
        rng = np.random.default_rng(nz)
        x = torch.from_numpy(rng.standard_normal((nrhs, m.n)) + 1j * rng.standard_normal((nrhs, m.n))).to("cuda")
        y = op.apply(x).cpu().numpy()
        monkeypatch.setenv("XTR_CONTRACT_KERNEL", "generic")
        g = op.apply(x).cpu().numpy()
        monkeypatch.delenv("XTR_CONTRACT_KERNEL")
        e = max(rel(y[r], g[r]) for r in range(nrhs))
        worst = max(worst, (e, nz))
        assert e < tol, (nz, e)
    print(f"nrhs {nrhs} {precision}: worst {worst[0]:.2e} at nz = {worst[1]}", flush=True)


@pytest.mark.parametrize("shape,nrhs", [((50, 60, 3), 2), ((48, 40, 8), 8), ((40, 30, 13), 1), ((24, 30, 17), 3),
                                        ((20, 24, 40), 2), ((16, 20, 47), 1), ((24, 24, 32), 4)])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 2e-6)])
def test_several_blocks_per_workgroup(oracle, torch_cuda, shape, nrhs, precision, tol):
    m, w, G, op = _op(oracle, shape, nrhs, precision, sum(shape))
    oop = oracle.Operator(m, G)
    oop.prepare("A", m.zeta(w).reshape(-1), m.zeta0(w))
    rng = np.random.default_rng(3)
    xs = rng.standard_normal((nrhs, m.n)) + 1j * rng.standard_normal((nrhs, m.n))
    y = op.apply(xs)
    errs = [rel(y[r], oop.apply(xs[r])) for r in {0, nrhs - 1}]
    print(f"{shape} nrhs {nrhs} {precision}: {max(errs):.2e}", flush=True)
    assert max(errs) < tol
