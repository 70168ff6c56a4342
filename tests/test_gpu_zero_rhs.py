"""A solve of a zero right-hand side is over when its norm is known: it applies the operator to nothing, neither alone
nor beside right-hand sides that do."""
import numpy as np
import pytest

from extreme_amd import cartesian_model as cm
from extreme_amd import xtreme as X

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("zeros,others", [(1, 0), (2, 0), (2, 1), (1, 2)])
def test_zero_right_hand_sides_cost_no_apply(torch_cuda, zeros, others):
    torch = torch_cuda
    n = zeros + others
    m = cm.small_model(8, 6, 4, contrast=30.0, seed=3)
    op = X.ConvolutionOperator(m, cm.omega_of(1.0), max_rhs=n)
    op.calculate_green_tensor()
    op.prepare_operator("A")
    rng = np.random.default_rng(1)
    x = torch.from_numpy(rng.standard_normal((n, m.n)) + 1j * rng.standard_normal((n, m.n))).to("cuda")
    b = x.clone()
    b[:zeros] = 0
    x0 = x.clone()
    op.set_profiling(True)
    s = X.AnomalyCurrentFgmresSolver(op)
    infos = [s.solve(b[0], x[0])] if n == 1 else s.solve_batch([b[r] for r in range(n)], [x[r] for r in range(n)])
    for r in range(zeros):
        i = infos[r]
        assert i.convergence_achieved and (i.number_of_iterations, i.matvecs, i.dot_products) == (0, 0, 1)
        assert torch.equal(x[r], x0[r])
    # applies of k right-hand sides, times k, are the applies of the solves that had work
    applied = sum(k * op.stage_times(k)[1] for k in range(1, n + 1))
    assert applied == sum(i.matvecs for i in infos[zeros:])
    assert op.stage_times(0)[1] == max([i.matvecs for i in infos[zeros:]], default=0)
    assert all(i.convergence_achieved and i.backward_error < 1e-8 for i in infos[zeros:])
