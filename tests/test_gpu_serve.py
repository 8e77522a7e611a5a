"""Serving loop on the GPU: admission by HBM footprint, continuous batching
(requests joining while others are mid-flight), isolation of each result,
and refusal of requests larger than the budget.

The clock is virtual (one unit per scheduling tick) so arrivals interleave
with running requests deterministically."""
import numpy as np
import pytest

from conftest import CFG1, cfg2_params
from test_gpu_api import build_problem, field_errors
from test_gpu_batch import P_A1, P_A3

pytestmark = pytest.mark.gpu

ISOLATION_RTOL = 1e-9     # per-field relative L2, served alone vs in the mix

# (mesh n, params, arrival tick, steps)
REQS = [(3, CFG1, 0, 3), (2, P_A3, 0, 2), (4, P_A1, 1, 4), (2, CFG1, 2, 2), (3, P_A3, 3, 1)]


class VClock:
    def __init__(self):
        self.t = 0.0

    def __call__(self):
        return self.t


def _requests(which):
    from waterscapes_amd.serve import Request
    out = []
    for i in which:
        n, params, arr, steps = REQS[i]
        out.append(Request(make_solver=lambda n=n, params=params:
                           build_problem(n, params, "fp64", False, T=10.0, dt=0.05)[1],
                           steps=steps, arrival=float(arr), rid=i))
    return out


def _serve(reqs, budget=200e9, **kw):
    """Synchronous set-up (setup_workers = 0), so that admission happens at
    the tick a request arrives and the schedule is deterministic."""
    from waterscapes_amd.serve import MPETServer
    clock = VClock()
    srv = MPETServer(hbm_budget=budget, precision="mixed", outer_tol=1e-11, clock=clock,
                     setup_workers=0, **kw)
    for r in reqs:
        srv.submit(r)
    concurrency = []
    while srv.busy():
        concurrency.append(srv.tick())          # instances stepped together
        clock.t += 1.0
    return srv, concurrency


def test_continuous_batching_and_isolation():
    srv, conc = _serve(_requests(range(len(REQS))))
    done = {r.rid: r for r in srv.finished}
    assert len(done) == len(REQS) and not any(r.refused for r in done.values())
    # requests arriving later joined while earlier ones were still running
    assert done[2].admitted > 0 and done[2].admitted < done[0].done
    assert max(conc) >= 3
    for r in done.values():
        assert r.steps_done == r.steps and len(r.niter) == r.steps and min(r.niter) > 0
    # each result is the same served alone
    for i in range(len(REQS)):
        alone, _ = _serve(_requests([i]))
        a = alone.finished[0]
        from waterscapes_amd.fem import MixedSpace
        from waterscapes_amd.mesh import UnitCubeMesh
        n, params = REQS[i][0], REQS[i][1]
        space = MixedSpace(UnitCubeMesh(n, n, n), params["J"])
        errs = field_errors(space, done[i].result, a.result)
        assert max(errs) <= ISOLATION_RTOL, (i, errs)


def test_srpt_policy_least_remaining_work_first():
    """With a tick quota of one unknown, each tick steps exactly one
    instance: the one with the least remaining work (steps left x DOFs), so
    requests finish in the order of their work; results equal those of the
    every-instance policy."""
    which = [0, 1, 2, 3]
    reqs = _requests(which)
    for r in reqs:
        r.arrival = 0.0
    srv, conc = _serve(reqs, tick_dofs=1)
    assert set(conc) == {1}
    work = {r.rid: r.steps * r.ndofs for r in srv.finished}
    order = [r.rid for r in sorted(srv.finished, key=lambda r: r.done)]
    assert order == sorted(which, key=lambda i: (work[i], i)), (order, work)
    ref_reqs = _requests(which)
    for r in ref_reqs:
        r.arrival = 0.0
    ref, conc_all = _serve(ref_reqs, policy="all")
    assert conc_all[0] == len(which)
    by = {r.rid: r.result for r in ref.finished}
    from waterscapes_amd.fem import MixedSpace
    from waterscapes_amd.mesh import UnitCubeMesh
    for r in srv.finished:
        n, params = REQS[r.rid][0], REQS[r.rid][1]
        space = MixedSpace(UnitCubeMesh(n, n, n), params["J"])
        assert max(field_errors(space, r.result, by[r.rid])) <= ISOLATION_RTOL, r.rid


def test_admission_by_footprint():
    from waterscapes_amd.serve import footprint_bytes
    reqs = _requests([0, 2, 3])
    # budget for one instance at a time: the others wait until memory frees
    s = reqs[1].make_solver()
    one = footprint_bytes(s.up_.function_space(), "mixed")
    del s
    srv, conc = _serve(reqs, budget=1.05 * one)
    assert max(conc) == 1
    assert all(not r.refused and r.steps_done == r.steps for r in srv.finished)
    assert srv.used == 0
    # a request larger than the whole budget is refused, the rest still run
    srv, conc = _serve(_requests([2, 1]), budget=0.5 * one)
    by = {r.rid: r for r in srv.finished}
    assert by[2].refused and by[2].result is None
    assert not by[1].refused and by[1].steps_done == REQS[1][3]


def test_footprint_estimate_bounds_allocation():
    import torch
    from waterscapes_amd.batch import MPETBatch
    from waterscapes_amd.serve import footprint_bytes
    torch.cuda.synchronize()
    base = torch.cuda.memory_allocated()
    s = build_problem(4, CFG1, "fp64", False, T=10.0, dt=0.05)[1]
    b = MPETBatch([s], precision="mixed")
    b.step()
    torch.cuda.synchronize()
    used = torch.cuda.memory_allocated() - base
    est = footprint_bytes(s.up_.function_space(), "mixed")
    b.close()
    # torch's allocations only (native workspaces are extra): the estimate
    # must cover them and not overshoot grossly
    assert 0.5 * used <= est <= 6.0 * used, (est, used)


@pytest.mark.parametrize("n,A,count,precision,limit", [
    (8, 4, 1, "mixed", None), (8, 4, 1, "mixed", 1 << 20), (8, 1, 3, "mixed", 1 << 23),
    (4, 2, 1, "fp64", None), (4, 2, 3, "fp64", 1 << 18)])
def test_dense_ends_stay_within_their_limit(n, A, count, precision, limit):
    """What a batch with dense ends holds more than one without (limit 0) is
    at most dense_held of its limit (torch's allocations)."""
    import gc
    import torch
    from waterscapes_amd.batch import MPETBatch
    from waterscapes_amd.levels import DENSE_TAIL_BYTES
    from waterscapes_amd.serve import dense_held
    w = torch.ones(64, 64, dtype=torch.float64, device="cuda")
    w @ w                                        # the BLAS workspace is the process's
    del w

    def used(limit):
        gc.collect()
        torch.cuda.synchronize()
        base = torch.cuda.memory_allocated()
        sol = [build_problem(n, cfg2_params(A), "fp64", False, T=10.0, dt=0.05)[1]
               for _ in range(count)]
        b = MPETBatch(sol, precision=precision, dense_bytes=limit)
        assert all(s.converged for s in b.step())
        gc.collect()
        torch.cuda.synchronize()
        out = torch.cuda.memory_allocated() - base
        b.close()
        return out
    bound = dense_held(DENSE_TAIL_BYTES if limit is None else limit, precision)
    assert used(limit) - used(0) <= bound


def test_dense_ends_take_what_the_budget_leaves():
    """A tight budget admits what it admitted without dense ends; they take
    what is left."""
    from waterscapes_amd import levels as lv
    from waterscapes_amd.serve import MPETServer, dense_held, footprint_bytes
    reqs = _requests([2])
    one = footprint_bytes(reqs[0].make_solver().up_.function_space(), "mixed")
    limits = []
    for budget in (float(one), one + 6e5, 1e9):
        srv = MPETServer(hbm_budget=budget, precision="mixed", outer_tol=1e-11,
                         setup_workers=0)
        r = _requests([2])[0]
        r.arrival = 0.0
        srv.submit(r)
        srv.tick()
        limits.append(srv.batch.dense_bytes)
        assert srv.used + dense_held(limits[-1]) <= budget
        srv.run()
        assert not r.refused and r.steps_done == r.steps
    assert limits == [0, 100000, lv.DENSE_TAIL_BYTES]


def test_setup_threads_overlap_ticks_and_keep_results():
    """With set-up threads (the default), a request whose set-up is slow
    does not hold up the others: ticks keep stepping the running instances
    while it is prepared, and every result equals the synchronous server's."""
    import time
    from waterscapes_amd.serve import MPETServer
    sync, _ = _serve(_requests([0, 2, 3]))
    ref = {r.rid: r.result for r in sync.finished}
    reqs = _requests([0, 2, 3])
    slow = reqs[1].make_solver

    def slow_make():
        time.sleep(1.0)                          # a long host set-up
        return slow()
    reqs[1].make_solver = slow_make
    for r in reqs:
        r.arrival = 0.0
    srv = MPETServer(hbm_budget=200e9, precision="mixed", outer_tol=1e-11, setup_workers=2)
    for r in reqs:
        srv.submit(r)
    ticks_while_preparing = 0
    while srv.busy():
        prep = bool(srv.preparing) or any(r._fp is not None and not r._fp.done()
                                          for r in srv.waiting)
        if srv.tick() and prep:
            ticks_while_preparing += 1
        elif not srv.active:
            time.sleep(1e-3)
    srv.close()
    assert ticks_while_preparing >= 1
    done = {r.rid: r for r in srv.finished}
    assert len(done) == 3 and all(r.steps_done == r.steps for r in done.values())
    from waterscapes_amd.fem import MixedSpace
    from waterscapes_amd.mesh import UnitCubeMesh
    for rid, r in done.items():
        n, params = REQS[rid][0], REQS[rid][1]
        space = MixedSpace(UnitCubeMesh(n, n, n), params["J"])
        assert max(field_errors(space, r.result, ref[rid])) <= ISOLATION_RTOL, rid
