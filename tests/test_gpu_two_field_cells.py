"""The two-field operator cell by cell (GPU): equal to the CSR matrix, with
Robin facets, masks and one to four networks; the solves equal the CSR
path's and the oracle's; replayed chunks equal single launches bit for bit.

Both forms of a row add at most ~600 FP64 products (600 eps = 1.3e-13 of
their absolute sum), and the cells' contributions cancel by less than a
factor of 10 in the assembled entries: 2e-12 of (|A| |x|), per block."""
import numpy as np
import pytest

from conftest import CFG1, cfg2_params
from test_gpu_two_field import build, field_errors, oracle_problem

pytestmark = pytest.mark.gpu

OP_RTOL = 2e-12
ACC_RTOL = 1e-8          # per-field relative L2 error vs the oracle
PATH_RTOL = 1e-9         # between two solves to krylov_rtol 1e-12


def _build(cells, monkeypatch, n, params, **kw):
    from waterscapes_amd import mpetsolver as M
    monkeypatch.setattr(M, "TWO_FIELD_CELLS", 1 if cells else 10**9)
    problem, solver, sym = build(n, params, **kw)
    eng = solver.engine()
    assert (getattr(eng.krylov, "cell_desc64", None) is not None) == cells
    return solver, sym, eng


@pytest.mark.parametrize("params,n,kw", [(CFG1, 3, {"facets": True}), (cfg2_params(1), 7, {}),
                                         (cfg2_params(4), 5, {})])
def test_operator_equals_csr(params, n, kw, monkeypatch):
    import torch
    solver, _, eng = _build(True, monkeypatch, n, params, **kw)
    s = eng.system
    rp, ci, v = (t.cpu().numpy() for t in s.csr)
    import scipy.sparse as sp
    A = sp.csr_matrix((v[: rp[-1]], ci[: rp[-1]], rp), shape=(s.n, s.n))
    dm = s.dmask.cpu().numpy().astype(bool)
    rng = np.random.default_rng(n)
    x, b = rng.standard_normal(s.n), rng.standard_normal(s.n)
    xd, bd = torch.as_tensor(x).cuda(), torch.as_tensor(b).cuda()
    bound = abs(A) @ abs(x)
    nu = 3 * s.nP2
    for got, want in ((s.cell_apply(xd, masked=False), A @ x),
                      (s.cell_apply(xd), np.where(dm, 0.0, A @ x)),
                      (s.cell_apply(xd, bd), np.where(dm, 0.0, b - A @ x))):
        d = abs(got.cpu().numpy() - want)
        assert d[:nu].max() <= OP_RTOL * bound[:nu].max()
        assert d[nu:].max() <= OP_RTOL * bound[nu:].max()


@pytest.mark.parametrize("params,facets", [(CFG1, True), (cfg2_params(1), False),
                                           (cfg2_params(4), False)])
def test_solves_equal_csr_and_oracle(params, facets, monkeypatch):
    out = []
    for cells in (True, False):
        solver, sym, eng = _build(cells, monkeypatch, 3, params, facets=facets, krylov_rtol=1e-12)
        ref = oracle_problem(solver, params, sym, 0.05, 1.0, 0.1, facets)
        x0 = solver.up_.vector().get_local().copy()
        out.append([up.vector().get_local().copy() for up, t in solver.solve()])
    space = solver.up_.function_space()
    want = [(x.copy(), t) for x, t in ref.solve_direct(x0)]
    assert len(out[0]) == len(out[1]) == len(want)
    for a, b, (z, _) in zip(*out, want):
        assert np.linalg.norm(a - b) <= PATH_RTOL * np.linalg.norm(b)
        assert max(field_errors(space, a, z)) <= ACC_RTOL


def test_replayed_chunks_equal_single_launches(monkeypatch):
    import torch
    from waterscapes_amd.solver import StepEngine
    solver, _, eng = _build(True, monkeypatch, 4, CFG1)
    cfg = solver._config()
    cfg.use_graphs = False
    plain = StepEngine(solver.problem, solver.up_.function_space(), 0.05,
                       solver.params["theta"], cfg)
    g = torch.Generator(device="cpu").manual_seed(1)
    for _ in range(3):
        b = torch.randn(eng.system.n, generator=g, dtype=torch.float64).cuda()
        x, y = torch.zeros_like(b), torch.zeros_like(b)
        eng.krylov.solve(b, x)
        (b * 2.0).sum().item()
        plain.krylov.solve(b, y)
        assert torch.equal(x, y)
