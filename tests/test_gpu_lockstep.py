"""Solves that run in step share their launches: a right-hand side that needs no work, or that fails, must not
change the others', and a handle must serve again after a failed solve."""
import numpy as np
import pytest

from extreme_amd import cartesian_model as cm
from extreme_amd import xtreme as X

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def problem(torch_cuda):
    torch = torch_cuda
    m = cm.small_model(12, 10, 5, contrast=30.0, seed=3)
    op = X.ConvolutionOperator(m, cm.omega_of(1.0), max_rhs=4)
    op.calculate_green_tensor()
    op.prepare_operator("A")
    rng = np.random.default_rng(1)
    b = torch.from_numpy(rng.standard_normal((4, m.n)) + 1j * rng.standard_normal((4, m.n))).to("cuda")
    return torch, op, b


def _solve(op, b, x):
    s = X.AnomalyCurrentFgmresSolver(op)
    return s.solve_batch([b[r] for r in range(len(b))], [x[r] for r in range(len(x))]), s.history


def test_each_equals_its_own_solve(problem):
    torch, op, b = problem
    b = b.clone()
    b[2] = 0                                   # converged at once, without an apply
    x = torch.zeros_like(b)
    x[1] = b[1]                                # another initial guess: another number of steps
    x0 = x.clone()
    infos, history = _solve(op, b, x)
    assert infos[2].convergence_achieved and infos[2].matvecs == 0 and infos[2].number_of_iterations == 0
    assert torch.equal(x[2], x0[2])
    for r in (0, 1, 3):
        y = x0[r].clone()
        one = X.AnomalyCurrentFgmresSolver(op)
        info = one.solve(b[r], y)
        assert torch.equal(x[r], y), r
        assert (infos[r].number_of_iterations, infos[r].matvecs, infos[r].dot_products) == (
            info.number_of_iterations, info.matvecs, info.dot_products)
        assert [h[1:] for h in history if h[0] == r] == [h[1:] for h in one.history]


def test_one_failing_right_hand_side(problem):
    torch, op, b = problem
    bad = b[:3].clone()
    bad[1, 7] = float("nan")
    x = torch.zeros_like(bad)
    with pytest.raises(X.XtrError, match="NaN or Inf"):
        _solve(op, bad, x)
    for r in (0, 2):                           # the others ran to their end
        y = torch.zeros_like(b[r])
        X.AnomalyCurrentFgmresSolver(op).solve(b[r], y)
        assert torch.equal(x[r], y)
    x = torch.zeros_like(b[:2])
    infos, _ = _solve(op, b[:2], x)            # and the handle serves again
    assert all(i.convergence_achieved and i.backward_error < 1e-8 for i in infos)
