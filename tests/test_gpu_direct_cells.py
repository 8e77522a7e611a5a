"""The direct path's FP64 MINRES on the cell-wise operator, from captured
iteration chunks (GPU): the fields of every step equal the CSR path's and
the oracle's direct solve, for one to four networks; the replayed chunks
give what iterations launched one by one give, bit for bit, over several
solves with other device work between them."""
import numpy as np
import pytest

from conftest import CFG1, cfg2_params
from test_gpu_api import build_problem, field_errors, oracle_steps

pytestmark = pytest.mark.gpu

ACC_RTOL = 1e-8          # per-field relative L2 error vs the oracle
PATH_RTOL = 1e-9         # between two solves to 1e-12 of the right-hand side


def _fields(params, cells, monkeypatch, n=3, **kw):
    from waterscapes_amd import solver as S
    monkeypatch.setattr(S, "DIRECT_CELLS", 1 if cells else 10**9)
    problem, solver, sym = build_problem(n, params, "fp64", True, T=0.15, dt=0.05, **kw)
    eng = solver.engine()
    assert (eng.krylov.csr_desc is None) == cells
    assert (eng.krylov.cell_desc64 is not None) == cells
    ref = oracle_steps(solver, params, sym, 0.05, 1.0, 0.15)     # from the initial state
    return solver, ref, [up.vector().get_local().copy() for up, t in solver.solve()]


@pytest.mark.parametrize("params", [CFG1, cfg2_params(1), cfg2_params(4)])
def test_cells_match_csr_and_oracle(params, monkeypatch):
    solver, ref, a = _fields(params, True, monkeypatch)
    _, _, b = _fields(params, False, monkeypatch)
    space = solver.up_.function_space()
    assert len(a) == len(b) == len(ref) == 3
    for x, y, (z, _) in zip(a, b, ref):
        assert np.linalg.norm(x - y) <= PATH_RTOL * np.linalg.norm(y)
        assert max(field_errors(space, x, z)) <= ACC_RTOL


@pytest.mark.parametrize("cells", [True, False])
def test_replayed_chunks_equal_single_launches(cells, monkeypatch):
    import torch
    from waterscapes_amd import solver as S
    monkeypatch.setattr(S, "DIRECT_CELLS", 1 if cells else 10**9)
    problem, solver, sym = build_problem(4, CFG1, "fp64", True, T=0.05, dt=0.05)
    eng = solver.engine()
    kr = eng.krylov
    assert kr.opt.use_graphs == 1
    plain_cfg = solver._config(True)
    plain_cfg.use_graphs = False
    plain = S.StepEngine(problem, solver.up_.function_space(), 0.05, solver.params["theta"],
                         plain_cfg)
    g = torch.Generator(device="cpu").manual_seed(1)
    for _ in range(3):
        b = torch.randn(eng.system.n, generator=g, dtype=torch.float64).cuda()
        x, y = torch.zeros_like(b), torch.zeros_like(b)
        kr.solve(b, x)
        (b * 2.0).sum().item()
        plain.krylov.solve(b, y)
        assert torch.equal(x, y)
