"""Error indicators for one to seven networks, with and without the staged copy
to the host and the sources read through LDS (GPU): random states on a box mesh
vs the oracle.
Every value is a sum of at most ~1e4 FP64 products of the same sign class
(1e4 eps = 2e-12): 1e-11 of the largest, as for two networks."""
import numpy as np
import pytest

from conftest import oracle_mesh
from oracle import mpet_oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-11


@pytest.mark.parametrize("A,staged,deg,with_g", [(1, False, 2, True), (3, True, 3, True),
                                                 (7, True, 2, True), (2, False, 3, False)])
def test_network_counts(A, staged, deg, with_g, monkeypatch):
    import torch
    from waterscapes_amd import MPETProblem, MPETSolver, Constant, Expression, BoxMesh
    from waterscapes_amd import adaptive
    monkeypatch.setattr(adaptive, "STAGED_CELLS", 0 if staged else 1 << 30)
    rng = np.random.default_rng(A)
    S = rng.uniform(0.1, 0.4, (A, A))
    S = np.triu(S, 1) + np.triu(S, 1).T
    params = dict(J=A, E=800.0, nu=0.3, alpha=tuple(rng.uniform(0.1, 0.9, A)),
                  c=tuple(rng.uniform(1e-2, 1e-1, A)), K=tuple(rng.uniform(0.05, 0.3, A)),
                  S=tuple(tuple(r) for r in S))
    mesh = BoxMesh((0.0, 0.0, 0.0), (1.0, 1.5, 0.7), 2, 3, 2)
    problem = MPETProblem(mesh, Constant(0.4), params=dict(params))
    # degree 2, and degree 3 without g (122 doubles a cell, the longest rows
    # that fit): the cell kernel reads the sources through LDS; else directly
    f_ = Expression(("x[0]*x[1]", "x[2]", "x[1]"), degree=deg)
    problem.f = Expression(("x[0]*x[1]", "x[2]", "x[0]*x[0]"), degree=deg)
    if with_g:
        problem.g = [Expression("x[1]", degree=1) for _ in range(A)]
    solver = MPETSolver(problem, dict(dt=0.05, theta=1.0, T=0.1))
    n = solver.up.function_space().dim()
    x, xp = rng.standard_normal(n), rng.standard_normal(n)
    solver.up.data.copy_(torch.as_tensor(x))
    solver.up_.data.copy_(torch.as_tensor(xp))
    est = adaptive.ErrorEstimator(problem, solver, f_)
    assert (est.stage is not None) == staged
    got = [est.indicators() for _ in range(2)]
    ref = O.error_indicators(
        oracle_mesh(solver.up.function_space()), params, x, xp, 0.05,
        f=lambda X, t: np.stack([X[:, 0] * X[:, 1], X[:, 2], X[:, 0] ** 2], 1),
        fp=lambda X, t: np.stack([X[:, 0] * X[:, 1], X[:, 2], X[:, 1]], 1),
        g=(lambda X, t: np.stack([X[:, 1]] * A, 1)) if with_g else None, f_degree=deg,
        g_degree=1, t=0.4)
    for a, b, c in zip(*got, ref):
        assert np.array_equal(a, b)
        assert np.abs(a - c).max() <= TOL * np.abs(c).max()
