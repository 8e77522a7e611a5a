"""Batched MPET stepping: many MPETTotalPressureSolver instances (uneven
meshes, network counts, parameters, boundary conditions and time steps)
advanced together on one GPU (csrc/batch.hip).

The reference steps one problem per MPETTotalPressureSolver
(mpet/mpettotalpressuresolver.py:456-502); a batch runs that per-instance
step for every active instance in one set of kernel launches:

  * each instance keeps its own device-resident system (assembled
    primitives, Dirichlet data, right-hand-side kernels) and its own host
    AMG setup, exactly as a single solver would;
  * the operator of all instances is applied cell by cell, in blocks that hold
    one instance's cells, or in small batches (BATCH_CELLS) packed into one
    block-diagonal structured operator (u rows of all instances first, then
    the pressure rows), and the hierarchies are concatenated level by level (instances
    with fewer levels are padded with identity-prolongation levels ending in
    their own coarsest matrix; the small ends are dense operators, one
    block per instance);
  * MINRES keeps one state per instance (each instance converges to its own
    tolerance with its own iteration count; finished instances are skipped).

Per-instance results equal the single-instance solver's to the solver
tolerance (not bitwise: padding and packing change rounding order).
"""
from __future__ import annotations

import ctypes as C
import time as _time

import numpy as np
import torch

from . import _lib, amg, levels as lv
from ._lib import check, ptr, MAXF
from .krylov import (MAXLEV, HierDesc, PrecDesc, SolveStats, SolverConfig, SolverOptions,
                     _pick_lpr, compact_level, set_level_degrees)
from .solver import StepEngine, extrapolated_guess, push_history


class BatchCoef(C.Structure):
    _fields_ = [("C", C.c_double * (MAXF * MAXF)), ("stiff", C.c_double * MAXF),
                ("st_base", C.c_int64), ("k11_base", C.c_int64), ("nnz11", C.c_int64),
                ("F", C.c_int32), ("pad", C.c_int32)]


class BatchOpDesc(C.Structure):
    _fields_ = [("ninst", C.c_int32), ("nP2", C.c_int32), ("nP1", C.c_int32),
                ("rp22", C.c_void_p), ("ci22", C.c_void_p), ("rp21", C.c_void_p),
                ("ci21", C.c_void_p), ("rp12", C.c_void_p), ("ci12", C.c_void_p),
                ("rp11", C.c_void_p), ("ci11", C.c_void_p), ("nnz22", C.c_int64),
                ("nnz21", C.c_int64), ("nnz12", C.c_int64), ("nnz11", C.c_int64),
                ("dtype", C.c_int32), ("Kuu", C.c_void_p), ("Dv", C.c_void_p),
                ("Dt", C.c_void_p), ("M1", C.c_void_p), ("St", C.c_void_p),
                ("p_inst", C.c_void_p), ("p_base", C.c_void_p), ("coef", C.c_void_p),
                ("dmask", C.c_void_p)]


class BatchLayout(C.Structure):
    _fields_ = [("ninst", C.c_int32), ("p2_off", C.c_void_p), ("p1_off", C.c_void_p),
                ("pd_off", C.c_void_p)]


class BatchCellDesc(C.Structure):
    _fields_ = [(k, C.c_int32) for k in ("nblk", "cells_per_block", "npart2", "npart1")] + \
        [(k, C.c_void_p) for k in ("blk_inst", "blk_cells", "node2", "node1", "geom64", "geom32",
                                   "mu", "bq2", "lrp2", "pe2", "lsl2", "bq1", "lrp1", "pe1",
                                   "lsl1", "inc2_rp", "inc1_rp")]


# Cells from which a batch's operator runs cell by cell: two launches either
# way, but a third of the bytes of the packed assembled values and more work a
# cell.  An iteration cell by cell / packed, us: four instances of 5,400 cells in
# all 82.9 / 78.3, 12,576 82.0 / 82.1, 17,820 94.2 / 92.5, 24,360 96.5 / 99.6,
# 41,904 134.6 / 146.7; 12 of 16,200 98.7 / 96.6, of 25,452 101.0 / 104.9; 32 of
# 20,736 126.6 / 122.2.
BATCH_CELLS = 20000


def _bind():
    L = _lib.lib()
    P = C.c_void_p
    for name, args in (("mpet_batch_set_cell_operator", [P, P]),
                       ("mpet_batch_create", [P, P, P, P, P, P, C.POINTER(C.c_void_p)]),
                       ("mpet_batch_destroy", [P]),
                       ("mpet_batch_solve", [P, P, P, P, P, P]),
                       ("mpet_batch_apply", [P, C.c_int, P, P, P, P]),
                       ("mpet_batch_precond_apply", [P, C.c_int, P, P, P])):
        fn = getattr(L, name)
        fn.argtypes = args
        fn.restype = C.c_int
    return L


def _prefix(sizes):
    out = np.zeros(len(sizes) + 1, dtype=np.int64)
    np.cumsum(np.asarray(sizes, dtype=np.int64), out=out[1:])
    return out


def _i32(a):
    a = np.asarray(a)
    if a.size and (a.max() >= 2**31 or a.min() < -2**31):
        raise ValueError("batch too large for 32-bit indices")
    return np.ascontiguousarray(a, dtype=np.int32)


def pad_levels(levels, cinv, depth):
    """The levels of one instance extended to `depth`: its coarsest level
    becomes an inner one with no matrix and a zero diagonal inverse (its
    smoothing steps leave 0 and then the correction untouched, its residual
    is the right-hand side) and passes everything through identity
    prolongators to the coarsest solve at the bottom, which therefore may be
    any operator, not only the exact inverse."""
    levels = [dict(lev) for lev in levels]
    last = levels[-1]
    n = last["n"]
    eye_rp = np.arange(n + 1, dtype=np.int64)
    eye_ci = np.arange(n, dtype=np.int32)
    eye_v = np.ones(n)
    none = dict(A_rp=np.zeros(n + 1, dtype=np.int64), A_ci=np.zeros(0, dtype=np.int32),
                A_v=np.zeros(0), dinv=np.zeros(n))
    while len(levels) < depth:
        levels[-1].update(nc=n, P_rp=eye_rp, P_ci=eye_ci, P_v=eye_v, R_rp=eye_rp, R_ci=eye_ci,
                          R_v=eye_v, **none)
        levels.append(dict(n=n, nc=0, A_rp=last["A_rp"], A_ci=last["A_ci"], A_v=last["A_v"],
                           dinv=last["dinv"], rho=last["rho"]))
    return levels, cinv


def csr_blockdiag(blocks):
    """Block-diagonal CSR of blocks (rp, ci, v, nrows, ncols) given as host
    arrays: row pointers int64, columns int32."""
    roff = _prefix([b[3] for b in blocks])
    coff = _prefix([b[4] for b in blocks])
    voff = _prefix([b[0][-1] for b in blocks])
    rp = np.concatenate([np.asarray(b[0][:-1], dtype=np.int64) + voff[k]
                         for k, b in enumerate(blocks)] + [voff[-1:]])
    ci = np.concatenate([np.asarray(b[1], dtype=np.int64) + coff[k]
                         for k, b in enumerate(blocks)])
    v = np.concatenate([np.asarray(b[2], dtype=np.float64) for b in blocks])
    return rp, _i32(ci), v, int(roff[-1]), int(coff[-1])


def pack_hierarchy(hiers, scales, skip_A0=False):
    """Concatenate instance hierarchies level by level (host arrays; the dense
    coarsest operators on the device where one of them is there).

    hiers: list of (levels, cinv) as returned by amg.setup_host; scales:
    per-instance factor s_k (the packed hierarchy approximates
    blockdiag(s_k A_k)^-1: matrices times s_k, inverses divided by s_k).
    Each level's diagonal inverse is also divided by its spectral-radius
    estimate so that one Chebyshev interval (rho = 1) fits every instance.
    skip_A0: leave out the level-0 matrix (the caller supplies it on the
    device).  Each level also carries grp, the instance of each of its rows.
    Returns (levels, coarse) with coarse = (inv, blk, off, ioff)."""
    depth = max(len(h[0]) for h in hiers)
    padded = [pad_levels(lv, ci, depth) for lv, ci in hiers]
    s = np.asarray(scales, dtype=np.float64)
    out = []
    for l in range(depth):
        lev_k = [p[0][l] for p in padded]
        rows = _prefix([lv["n"] for lv in lev_k])
        d = dict(n=int(rows[-1]), rho=1.0, nc=0,
                 dinv=np.concatenate([lv["dinv"] / (s[k] * lv["rho"])
                                      for k, lv in enumerate(lev_k)]),
                 grp=np.repeat(np.arange(len(lev_k), dtype=np.int32), np.diff(rows)))
        if not (l == 0 and skip_A0):
            d["A_rp"], d["A_ci"], d["A_v"], _, _ = csr_blockdiag(
                [(lv["A_rp"], lv["A_ci"], lv["A_v"] * s[k], lv["n"], lv["n"])
                 for k, lv in enumerate(lev_k)])
        if l < depth - 1:
            P = csr_blockdiag([(lv["P_rp"], lv["P_ci"], lv["P_v"], lv["n"], lv["nc"])
                               for lv in lev_k])
            R = csr_blockdiag([(lv["R_rp"], lv["R_ci"], lv["R_v"], lv["nc"], lv["n"])
                               for lv in lev_k])
            d.update(nc=P[4], P_rp=P[0], P_ci=P[1], P_v=P[2], R_rp=R[0], R_ci=R[1], R_v=R[2])
        out.append(d)
    sizes = [p[0][-1]["n"] for p in padded]
    off = _prefix(sizes)
    dev = next((p[1].device for p in padded if torch.is_tensor(p[1])), None)
    if dev is not None:
        inv = torch.cat([(torch.as_tensor(p[1]).to(dev, torch.float64) / s[k]).reshape(-1)
                         for k, p in enumerate(padded)])
    else:
        inv = np.concatenate([(np.asarray(p[1]) / s[k]).reshape(-1)
                              for k, p in enumerate(padded)])
    ioff = _prefix([n * n for n in sizes])
    blk = np.repeat(np.arange(len(sizes), dtype=np.int32), sizes)
    return out, (inv, blk, _i32(off), ioff)


def batch_engine(solver, precision="mixed", system=None):
    """The batch-ready device state of one solver (assembled system, Dirichlet
    data, RHS kernels, host AMG hierarchies), created once and kept on the
    solver, so that re-packing a batch never repeats assembly or AMG setup.
    system: its DeviceSystem, already assembled (by a batched assembly)."""
    eng = getattr(solver, "_engine", None)
    if eng is not None and getattr(eng, "batched", False) and eng.config.mode == precision:
        return eng
    p = solver.params
    cfg = SolverConfig(mode=precision, p0_weight=p["p0_weight"])
    eng = StepEngine(solver.problem, solver.up_.function_space(), p["dt"], p["theta"], cfg,
                     p["device"], batched=True, system=system)
    solver._engine = eng
    return eng


def build_engines(solvers, precision="mixed", workers=None):
    """batch_engine of every solver.  Instances that have no engine yet get
    their systems assembled together (one launch per colour index for all
    of them, device.assemble_batch) and are then set up concurrently by a
    pool of host threads (their hierarchy setups run in native code without
    the interpreter lock, with the host cores split among the workers), each
    worker enqueuing its device work on a stream of its own and
    synchronising it before the engine is used."""
    import concurrent.futures as cf
    import os
    import threading
    from .device import assemble_batch
    from .solver import batch_system
    todo = [s for s in solvers if not (getattr(s, "_engine", None) is not None
                                       and getattr(s._engine, "batched", False)
                                       and s._engine.config.mode == precision)]
    systems = {}
    if len(todo) > 1:
        for s in todo:
            systems[id(s)] = batch_system(s.problem, s.up_.function_space(), s.params["dt"],
                                          s.params["theta"], s.params["device"],
                                          assemble=False)
        assemble_batch(list(systems.values()))
    ncpu = len(os.sched_getaffinity(0))
    workers = workers or max(1, min(8, len(todo), ncpu // 2))
    if workers > 1 and len(todo) > 1:
        local = threading.local()
        dev = torch.device(solvers[0].params["device"])

        def work(s):
            if not hasattr(local, "stream"):
                local.stream = torch.cuda.Stream(device=dev)
                amg.set_host_threads(max(1, ncpu // workers))
            with torch.cuda.stream(local.stream):
                e = batch_engine(s, precision, systems.get(id(s)))
            local.stream.synchronize()
            return e
        with cf.ThreadPoolExecutor(max_workers=workers) as ex:
            list(ex.map(work, todo))
    return [batch_engine(s, precision, systems.get(id(s))) for s in solvers]


class MPETBatch:
    """Advance many MPETTotalPressureSolver instances together.

    solvers: MPETTotalPressureSolver objects (each with its own problem and
    params); their "precision" is overridden by `precision` ("mixed" or
    "fp64").  The solvers' up_ / up become views into the batch's packed
    state, so initial conditions set on them before construction are kept
    and results are read from them as usual.  dense_bytes: most bytes of the
    dense ends of each of the two packed hierarchies (default
    levels.DENSE_TAIL_BYTES).
    """

    def __init__(self, solvers, precision="mixed", rtol=1e-10, outer_tol=3e-11,
                 inner_rtol=1e-6, maxit=5000, max_outer=30, check_every=10, use_graphs=True,
                 extrapolate=None, extrapolate_order=4, autotune=False, dense_bytes=None):
        if not torch.cuda.is_available():
            raise RuntimeError("MPETBatch needs a GPU (no CPU fallback)")
        if precision not in ("mixed", "fp64"):
            raise ValueError("precision must be 'mixed' or 'fp64'")
        self.solvers = list(solvers)
        if not self.solvers:
            raise ValueError("empty batch")
        self.precision = precision
        # initial guess extrapolated in time from u_n and the previous states
        # (polynomial degree extrapolate_order; the mixed path's outer
        # tolerance bounds the error independently of the guess)
        self.extrapolate = (precision == "mixed") if extrapolate is None else bool(extrapolate)
        self.ex_order = int(extrapolate_order)
        self.K = K = len(self.solvers)
        dev = torch.device(self.solvers[0].params["device"])
        self.device = dev
        for s in self.solvers:
            if str(torch.device(s.params["device"])) != str(dev):
                raise ValueError("all instances of a batch must be on one device")
        self.engines = build_engines(self.solvers, precision)
        # bytes of the packed dense ends of each of the two hierarchies
        self.dense_bytes = lv.DENSE_TAIL_BYTES if dense_bytes is None else int(dense_bytes)
        self.keep = []
        self.cells = sum(e.space.mesh.num_cells() for e in self.engines) >= BATCH_CELLS
        self._layout()
        self._pack_operator()
        self._pack_preconditioner()
        L = _bind()
        self.opt = SolverOptions({"fp64": 0, "mixed": 1}[precision], 0, rtol, maxit,
                                 check_every, 1 if use_graphs else 0, outer_tol, inner_rtol,
                                 max_outer)
        h = C.c_void_p()
        pc = C.byref(self.prec)
        check(L.mpet_batch_create(C.byref(self.op64),
                                  C.byref(self.op32) if self.op32 is not None else None,
                                  C.byref(self.layout), pc if precision == "fp64" else None,
                                  pc if precision == "mixed" else None, C.byref(self.opt),
                                  C.byref(h)))
        self.handle = h
        if self.cells:
            self.cell_desc = self._pack_cells()
            check(L.mpet_batch_set_cell_operator(h, C.byref(self.cell_desc)))
        self._state_views()
        self.stats = None
        self.tuning = None
        if autotune:
            self.autotune()

    def autotune(self, cache=None):
        """Lanes per row of the packed hierarchies' level SpMMs picked by
        the autotuner (waterscapes_amd/autotune.py) and applied to the
        handle; the packed operator keeps its fixed shapes."""
        from . import autotune as at
        dt = 0 if self.precision == "fp64" else 1
        out = {}
        for name, nc in (("u", 3), ("p", 1)):
            levels, devs = self.hier_levels[name]

            def rule(l, which, levels=levels, devs=devs, nc=nc):
                lev, ld = levels[l], devs[l]
                if which == "A":
                    return _pick_lpr(ld["A_ci"].numel() / max(lev["n"], 1), nc, lev["n"])
                nnzp = ld["P_ci"].numel()
                if which == "P":
                    return _pick_lpr(nnzp / max(lev["n"], 1), nc, lev["n"])
                return _pick_lpr(nnzp / max(lev["nc"], 1), nc, lev["nc"])
            out[name] = at.tune_hierarchy(levels, devs, nc, dt, rule,
                                          self.mask0 if name == "u" else None, cache)
        at.apply_tuning(self.handle, dt, u=out["u"], p=out["p"], batch=True)
        self.tuning = {"u_levels": out["u"], "p_levels": out["p"]}
        return self.tuning

    # -- layout and packing ----------------------------------------------------
    def _layout(self):
        sys_ = [e.system for e in self.engines]
        self.p2_off = _prefix([s.nP2 for s in sys_])
        self.p1_off = _prefix([s.nP1 for s in sys_])
        self.pd_off = _prefix([s.F * s.nP1 for s in sys_])
        self.n_off = _prefix([s.n for s in sys_])          # instance-major offsets
        self.nP2 = int(self.p2_off[-1])
        self.nP1 = int(self.p1_off[-1])
        self.nu = 3 * self.nP2
        self.n = self.nu + int(self.pd_off[-1])
        if self.n >= 2**31:
            raise ValueError("batch exceeds 2^31 DOFs")
        self.layout = BatchLayout(self.K, self.p2_off.ctypes.data, self.p1_off.ctypes.data,
                                  self.pd_off.ctypes.data)
        # packed index -> instance-major index
        perm = np.empty(self.n, dtype=np.int64)
        for k, s in enumerate(sys_):
            base = self.n_off[k]
            perm[3 * self.p2_off[k]:3 * self.p2_off[k + 1]] = base + np.arange(s.nu)
            p0 = self.nu + self.pd_off[k]
            perm[p0:p0 + s.F * s.nP1] = base + s.nu + np.arange(s.F * s.nP1)
        self.perm = torch.as_tensor(perm).to(self.device)

    def _pack_operator(self):
        dev = self.device
        sys_ = [e.system for e in self.engines]
        i32 = torch.int32
        nz = {k: _prefix([s.nnz[k] for s in sys_]) for k in ("22", "21", "12", "11")}
        self.nnz_off = nz
        pats = {}
        for kind in ("22", "21", "12", "11"):
            rps, cis = [], []
            for k, s in enumerate(sys_):
                rp, ci = s.pat_dev[kind]
                rps.append(rp[:-1].to(torch.int64) + int(nz[kind][k]))
                if kind in ("22", "12"):     # columns are P2 nodes
                    cis.append(ci.to(torch.int64) + int(self.p2_off[k]))
                else:                        # columns are P1 nodes -> packed p_0 DOF
                    cis.append(ci.to(torch.int64) * s.F + int(self.nu + self.pd_off[k]))
            rps.append(torch.tensor([int(nz[kind][-1])], dtype=torch.int64, device=dev))
            rp = torch.cat(rps)
            ci = torch.cat(cis)
            if int(rp[-1]) >= 2**31 or (ci.numel() and int(ci.max()) >= 2**31):
                raise ValueError("batch too large for 32-bit pattern indices")
            pats[kind] = (rp.to(i32), ci.to(i32))
        self.pats = pats
        # per-P1-node instance and packed p_0 DOF
        p_inst = np.repeat(np.arange(self.K, dtype=np.int32), np.diff(self.p1_off))
        p_base = np.concatenate([self.nu + self.pd_off[k] + s.F * np.arange(s.nP1)
                                 for k, s in enumerate(sys_)])
        self.p_inst = torch.as_tensor(p_inst).to(dev)
        self.p_base = torch.as_tensor(_i32(p_base)).to(dev)
        # per-instance coefficients
        st_base = _prefix([s.A * s.nnz["11"] for s in sys_])
        coefs = (BatchCoef * self.K)()
        for k, s in enumerate(sys_):
            c = coefs[k]
            for f in range(s.F):
                for g in range(s.F):
                    c.C[f * MAXF + g] = float(s.Cm[f, g])
                c.stiff[f] = float(s.Cs[f])
            c.st_base = int(st_base[k])
            c.k11_base = int(nz["11"][k])
            c.nnz11 = int(s.nnz["11"])
            c.F = s.F
        raw = np.frombuffer(coefs, dtype=np.uint8).copy()
        self.coef_dev = torch.as_tensor(raw).to(dev)
        # Dirichlet mask (packed)
        m = torch.cat([s.dmask[:s.nu] for s in sys_] + [s.dmask[s.nu:] for s in sys_])
        self.dmask = m.contiguous()
        self.op64 = self._pack_values(0, st_base)
        self.op32 = self._pack_values(1, st_base) if self.precision == "mixed" else None

    def _pack_values(self, dtype, st_base):
        """Structure-of-arrays values of every instance in one packed array
        per primitive (strides = packed nonzero counts)."""
        dev = self.device
        tdt = torch.float64 if dtype == 0 else torch.float32
        sys_ = [e.system for e in self.engines]
        nz = self.nnz_off
        L = _lib.lib()
        sptr = _lib.stream_ptr()
        # cell by cell, only the P1 x P1 block is read from assembled values
        prims = (("M1", "11", 1),) if self.cells else \
            (("Kuu", "22", 9), ("Dv", "21", 3), ("Dt", "12", 3), ("M1", "11", 1))
        vals = dict.fromkeys(("Kuu", "Dv", "Dt"))
        for name, kind, ncomp in prims:
            tot = int(nz[kind][-1])
            out = torch.empty(ncomp * tot, dtype=tdt, device=dev)
            view = out.view(ncomp, tot)
            for k, s in enumerate(sys_):
                src = s.prim_t[name]
                n = src.numel() // ncomp
                tmp = torch.empty(ncomp * n, dtype=tdt, device=dev)
                check(L.mpet_soa_convert(dtype, ptr(src), ncomp, n, ptr(tmp), sptr))
                view[:, int(nz[kind][k]):int(nz[kind][k]) + n].copy_(tmp.view(ncomp, n))
                del tmp
            vals[name] = out
        vals["St"] = torch.cat([s.prim_t["St"].to(tdt) for s in sys_]) if sys_ else None
        assert vals["St"].numel() == int(st_base[-1])
        self.keep.append(vals)
        p = self.pats
        return BatchOpDesc(self.K, self.nP2, self.nP1, ptr(p["22"][0]), ptr(p["22"][1]),
                           ptr(p["21"][0]), ptr(p["21"][1]), ptr(p["12"][0]), ptr(p["12"][1]),
                           ptr(p["11"][0]), ptr(p["11"][1]), int(nz["22"][-1]),
                           int(nz["21"][-1]), int(nz["12"][-1]), int(nz["11"][-1]), dtype,
                           ptr(vals["Kuu"]), ptr(vals["Dv"]), ptr(vals["Dt"]), ptr(vals["M1"]),
                           ptr(vals["St"]), ptr(self.p_inst), ptr(self.p_base),
                           ptr(self.coef_dev), ptr(self.dmask))

    def _pack_cells(self):
        """The instances' cell-wise tables (DeviceSystem.cell_op) packed into
        one set (MpetBatchCellDesc)."""
        dev = self.device
        sys_ = [e.system for e in self.engines]
        B = sys_[0].CELLS_PER_BLOCK
        ops = [s.cell_op() for s in sys_]
        nblk = [(o["nC"] + B - 1) // B for o in ops]
        total = B * sum(nblk)

        def tables(kind, width, node_of, inc_len):
            node = torch.zeros(width, total, dtype=torch.int32, device=dev)
            out = {k: [] for k in ("bq", "lrp", "pe", "rp", "lsl")}
            parts = slots = at = 0
            for k, (s, o) in enumerate(zip(sys_, ops)):
                t = o[kind]
                node[:, at:at + o["nC"]] = node_of(k, t["node"].view(width, -1))
                for name, off in (("bq", parts), ("lrp", slots), ("rp", parts)):
                    v = t[name].long() + off
                    out[name].append(v if k == self.K - 1 else v[:-1])
                out["pe"].append(t["pe"].long() + parts)
                out["lsl"].append(t["lsl"])
                parts += t["npart"]
                slots += t["lsl"].numel()
                at += nblk[k] * B
            if max(3 * parts, slots) >= 2**31:
                raise ValueError("batch too large for 32-bit cell tables")
            r = {n: torch.cat(v) for n, v in out.items()}
            r = {n: v if n == "lsl" else v.to(torch.int32) for n, v in r.items()}
            assert r["rp"].numel() == inc_len + 1
            return node, r, parts
        n2, t2, np2 = tables("p2", 10, lambda k, t: t + int(self.p2_off[k]), self.nP2)
        n1, t1, np1 = tables("p1", 4, lambda k, t: t * sys_[k].F
                             + int(self.nu + self.pd_off[k]), self.nP1)
        geom = torch.zeros(10, total, dtype=torch.float64, device=dev)
        blk_cells, at = [], 0
        for s, o, nb in zip(sys_, ops, nblk):
            geom[:, at:at + o["nC"]] = s.cell_geom64().view(10, -1)
            blk_cells += [min(B, o["nC"] - B * i) for i in range(nb)]
            at += nb * B
        geom32 = geom.float() if self.precision == "mixed" else None
        inst = torch.as_tensor(np.repeat(np.arange(self.K, dtype=np.int32), nblk)).to(dev)
        cells = torch.as_tensor(np.asarray(blk_cells, dtype=np.int32)).to(dev)
        mu = np.array([s.mu for s in sys_], dtype=np.float64)
        self.keep += [n2, n1, t2, t1, geom, geom32, inst, cells, mu]
        return BatchCellDesc(sum(nblk), B, np2, np1, ptr(inst), ptr(cells), ptr(n2), ptr(n1),
                             ptr(geom), ptr(geom32), ptr(mu),
                             *(ptr(t2[k]) for k in ("bq", "lrp", "pe", "lsl")),
                             *(ptr(t1[k]) for k in ("bq", "lrp", "pe", "lsl")), ptr(t2["rp"]),
                             ptr(t1["rp"]))

    def _upload_hier(self, h, levels, coarse, params, mask0, nc, level0=None):
        dev = self.device
        tdt = torch.float64 if self.precision == "fp64" else torch.float32
        keep = []
        devs = []                   # per level: the device arrays (autotuner)
        h.nlev = len(levels)
        if h.nlev > MAXLEV:
            raise ValueError("hierarchy too deep")
        for l, lev in enumerate(levels):
            L = h.lev[l]
            ld = {}
            devs.append(ld)
            L.n = lev["n"]
            L.nc = lev["nc"]
            if l == 0 and level0 is not None:
                rp, ci, v = level0
            else:
                rp = torch.as_tensor(_i32(lev["A_rp"])).to(dev)
                ci = torch.as_tensor(lev["A_ci"]).to(dev)
                v = torch.as_tensor(lev["A_v"]).to(dev, tdt)
            dinv = torch.as_tensor(lev["dinv"]).to(dev, tdt)
            grp = torch.as_tensor(_i32(lev["grp"])).to(dev)
            keep += [rp, ci, v, dinv, grp]
            ld.update(A_rp=rp, A_ci=ci, A_v=v, dinv=dinv, grp=grp)
            L.A_rp, L.A_ci, L.A_v, L.dinv = ptr(rp), ptr(ci), ptr(v), ptr(dinv)
            L.grp = ptr(grp)
            if "A_v16" in lev:
                keep += [lev["A_v16"], lev["A_dci"]]
                ld.update(A_v16=lev["A_v16"], A_dci=lev["A_dci"], vscale=lev["vscale"])
                L.A_v16, L.A_dci, L.A_vscale = ptr(lev["A_v16"]), ptr(lev["A_dci"]), lev["vscale"]
            L.rho = lev["rho"]
            L.lpr = _pick_lpr(ci.numel() / max(lev["n"], 1), nc, lev["n"])
            if lev["nc"]:
                arrs = []
                for k in ("P", "R"):
                    a = (torch.as_tensor(_i32(lev[k + "_rp"])).to(dev),
                         torch.as_tensor(lev[k + "_ci"]).to(dev),
                         torch.as_tensor(lev[k + "_v"]).to(dev, tdt))
                    arrs.append(a)
                    keep += list(a)
                (L.P_rp, L.P_ci, L.P_v), (L.R_rp, L.R_ci, L.R_v) = \
                    [tuple(ptr(t) for t in a) for a in arrs]
                ld.update(P_rp=arrs[0][0], P_ci=arrs[0][1], P_v=arrs[0][2], R_rp=arrs[1][0],
                          R_ci=arrs[1][1], R_v=arrs[1][2])
                nnzp = arrs[0][1].numel()
                L.lprP = _pick_lpr(nnzp / max(lev["n"], 1), nc, lev["n"])
                L.lprR = _pick_lpr(nnzp / max(lev["nc"], 1), nc, lev["nc"])
        lv.add_fused(devs, levels, params, 0 if self.precision == "fp64" else 1, mask0)
        for l, ld in enumerate(devs):
            lv.describe_fused(h.lev[l], ld, levels[l]["n"], levels[l]["nc"], nc)
        inv, blk, off, ioff = coarse
        cinv = torch.as_tensor(inv).to(dev, tdt)
        cblk = torch.as_tensor(blk).to(dev)
        coff = torch.as_tensor(off).to(dev)
        cioff = torch.as_tensor(ioff).to(dev)
        keep += [cinv, cblk, coff, cioff]
        h.coarse_inv = ptr(cinv)
        h.coarse_blk, h.coarse_off, h.coarse_ioff = ptr(cblk), ptr(coff), ptr(cioff)
        h.degree = params.smoother_degree
        set_level_degrees(h, params)
        h.eig_ratio = params.eig_ratio
        h.eig_safety = params.eig_safety
        h.scale = 1.0
        h.mask0 = ptr(mask0) if mask0 is not None else None
        self.keep.append(keep)
        return devs

    def _pack_preconditioner(self):
        dev = self.device
        tdt = torch.float64 if self.precision == "fp64" else torch.float32
        kry = [e.krylov for e in self.engines]
        sys_ = [e.system for e in self.engines]
        # displacement block: scalar P2 Laplacian hierarchies scaled by mu_k
        mus = [s.mu for s in sys_]
        # the small end of every hierarchy as one dense operator per instance
        # (levels.py), all instances' together within the byte limit
        rows = lv.dense_rows(8 if self.precision == "fp64" else 4,
                             self.dense_bytes // self.K)
        cut = [k.dense_tails(rows, 0 if self.precision == "fp64" else 1) for k in kry]
        ulev, ucoarse = pack_hierarchy([c[0] for c in cut], mus, skip_A0=True)
        lap0 = torch.cat([s.prim_t["Lap"] * s.mu for s in sys_]).to(tdt)
        level0 = (self.pats["22"][0], (torch.cat([s.pat_dev["22"][1].to(torch.int64)
                                                  + int(self.p2_off[k])
                                                  for k, s in enumerate(sys_)])).to(torch.int32),
                  lap0)
        self.mask0 = torch.cat([k.mask0 for k in kry]).contiguous()
        if self.precision == "mixed" and kry[0].cfg.compact_level0:
            # half-precision finest level, as for one instance
            c = compact_level(level0[:2], torch.cat([s.prim_t["Lap"] * s.mu for s in sys_]))
            if c is not None:
                ulev[0].update(c)
        # pressure blocks: field-major block-diagonal hierarchies, scale 1
        plev, pcoarse = pack_hierarchy([c[1] for c in cut], [1.0] * self.K)
        pmap = np.concatenate([self.pd_off[k] + (np.arange(s.F)[None, :] * s.nP1
                                                 + np.arange(s.nP1)[:, None]).reshape(-1)
                               for k, s in enumerate(sys_)])
        self.pmap = torch.as_tensor(_i32(pmap)).to(dev)
        d = PrecDesc()
        cfg = kry[0].cfg
        udev = self._upload_hier(d.u, ulev, ucoarse, cfg.amg, self.mask0, 3, level0=level0)
        pdev = self._upload_hier(d.p, plev, pcoarse, cfg.pamg, None, 1)
        self.hier_levels = {"u": (ulev, udev), "p": (plev, pdev)}
        d.nP1 = int(self.pd_off[-1])
        d.F = 1
        d.pmap = ptr(self.pmap)
        self.prec = d
        self.hier_depth = (len(ulev), len(plev))

    def _state_views(self):
        """Instance-major right-hand side and state buffers; each engine's b
        and each solver's up_ / up become views into them."""
        dev = self.device
        f64 = torch.float64
        self.B_i = torch.zeros(self.n, dtype=f64, device=dev)
        self.X_i = torch.zeros(self.n, dtype=f64, device=dev)
        self.Xprev_i = torch.zeros(self.n, dtype=f64, device=dev)
        self.Bp = torch.empty(self.n, dtype=f64, device=dev)
        self.Xp = torch.empty(self.n, dtype=f64, device=dev)
        for k, (s, e) in enumerate(zip(self.solvers, self.engines)):
            a, b = int(self.n_off[k]), int(self.n_off[k + 1])
            self.Xprev_i[a:b].copy_(s.up_.data)
            self.X_i[a:b].copy_(s.up.data)
            s.up_.data = self.Xprev_i[a:b]
            s.up.data = self.X_i[a:b]
            e.b = self.B_i[a:b]
        self.t = [float(s.problem.time) for s in self.solvers]

    # -- operators (tests and diagnostics) -------------------------------------
    def pack(self, x_inst):
        """Instance-major vector -> packed numbering."""
        return x_inst[self.perm]

    def unpack(self, x_packed):
        out = torch.empty_like(x_packed)
        out[self.perm] = x_packed
        return out

    def apply(self, xp, b=None, dtype=0):
        y = torch.empty_like(xp)
        check(_bind().mpet_batch_apply(self.handle, dtype, ptr(xp), ptr(b), ptr(y),
                                       _lib.stream_ptr()))
        return y

    def precond(self, rp, dtype=None):
        dtype = (0 if self.precision == "fp64" else 1) if dtype is None else dtype
        z = torch.empty_like(rp)
        check(_bind().mpet_batch_precond_apply(self.handle, dtype, ptr(rp), ptr(z),
                                               _lib.stream_ptr()))
        return z

    # -- time stepping -----------------------------------------------------------
    def step(self, active=None, raise_on_fail=True):
        """One implicit step of every instance k with active[k] (default:
        all): the reference's per-step sequence (:461-494) for each, one
        batched solve for all.  Advances each instance's time; returns the
        per-instance SolveStats (zeros for inactive instances).  An instance
        that does not converge (status 3) or breaks down (NaN, status 4)
        raises MpetError (its .stats the per-instance stats) after every
        instance's result is stored; with raise_on_fail=False those two
        statuses return the stats instead."""
        act = np.ones(self.K, dtype=np.int32) if active is None else \
            np.asarray(active, dtype=np.int32).copy()
        t_next = list(self.t)
        for k in np.nonzero(act)[0]:
            e, s = self.engines[k], self.solvers[k]
            t_next[k] = e.assemble_rhs(s.up_.data, self.t[k])
            x = s.up.data
            extrapolated_guess(e.hist if self.extrapolate else [], self.ex_order, s.up_.data, x)
            if e.bc_dofs.numel():
                g = torch.as_tensor(e.bc_values(None)).to(self.device)
                x.index_copy_(0, e.bc_dofs, g)
        torch.index_select(self.B_i, 0, self.perm, out=self.Bp)
        torch.index_select(self.X_i, 0, self.perm, out=self.Xp)
        stats = (SolveStats * self.K)()
        rc = _bind().mpet_batch_solve(self.handle, ptr(self.Bp), ptr(self.Xp),
                                      act.ctypes.data, stats, _lib.stream_ptr())
        self.stats = stats
        # the other instances' solutions are valid whatever the status: keep
        # them, then report (stats[k].converged == 0 names the failed ones)
        self.X_i.index_copy_(0, self.perm, self.Xp)
        for k in np.nonzero(act)[0]:
            self.t[k] = t_next[k]
        if rc != 0 and (raise_on_fail or rc not in (3, 4)):
            try:
                check(rc)
            except _lib.MpetError as err:
                err.stats = stats
                raise
        return stats

    def commit(self, active=None):
        """up_ <- up for the stepped instances (the generator's update after
        its yield, :497-499) and their time Constants to t_{n+1}."""
        ks = range(self.K) if active is None else np.nonzero(np.asarray(active))[0]
        if self.extrapolate:
            for k in ks:
                push_history(self.engines[k].hist, self.ex_order, self.solvers[k].up_.data)
        if active is None:
            self.Xprev_i.copy_(self.X_i)
        else:
            for k in ks:
                self.solvers[k].up_.data.copy_(self.solvers[k].up.data)
        for k in ks:
            self.solvers[k].problem.time.assign(self.t[k])

    def solve(self):
        """Generator: steps every instance until its own T (each instance's
        loop condition t < T - 1e-9 of :456).  Yields (stepped, stats) per
        batched step, stepped = indices of the instances advanced; each
        solver's up holds its new state during the yield and up_ is updated
        after it, as in the single-instance generator."""
        Ts = [float(s.params["T"]) for s in self.solvers]
        for s in self.solvers:
            s.solver_monitor.setdefault("niter", [])
            s.solver_monitor.setdefault("outer", [])
            s.solver_monitor.setdefault("residual", [])
        while True:
            act = np.array([1 if self.t[k] < Ts[k] - 1e-9 else 0 for k in range(self.K)],
                           dtype=np.int32)
            if not act.any():
                return
            stats = self.step(act)
            for k in np.nonzero(act)[0]:
                m = self.solvers[k].solver_monitor
                m["niter"].append(int(stats[k].inner_iterations))
                m["outer"].append(int(stats[k].outer_iterations))
                m["residual"].append(float(stats[k].residual_norm))
            yield np.nonzero(act)[0], stats
            self.commit(act if not act.all() else None)

    def close(self):
        if getattr(self, "handle", None):
            torch.cuda.synchronize()
            _bind().mpet_batch_destroy(self.handle)
            self.handle = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass
