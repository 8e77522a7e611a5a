"""Fused residual / restriction and prolongation / smoothing of the AMG
levels (waterscapes_amd/levels.py, csrc/amg_cycle.h).

* CPU: W and Q equal the sparse products they stand for, with Dirichlet rows
  held at zero and with levels that carry no matrix (FP64 round-off); the
  sliced copies hold exactly the matrix.
* GPU: the block preconditioner with the fused transfers equals the numpy
  restatement's separate steps, in FP64 and FP32, on hierarchies of several
  sparse levels: joint launches of both cycles (no level sliced), separate
  ones with the large levels or all of them on one thread per row, degrees 1
  to 3, small and ordinary meshes."""
import numpy as np
import pytest
import scipy.sparse as sp

from test_batch_pack import _laplacian


def _host_values(rows, cols, X, Y):
    import torch
    nm = max(Y[0].numel() - 1, 1)

    def dense(t, m):
        return sp.csr_matrix((t[2].numpy(), t[1].numpy(), t[0].numpy()),
                             shape=(t[0].numel() - 1, m)).toarray()
    C = dense(X, nm) @ dense(Y, int(cols.max()) + 1)
    return torch.as_tensor(C[rows.numpy(), cols.numpy()])


@pytest.mark.parametrize("degree", [1, 3])
@pytest.mark.parametrize("masked,empty", [(False, False), (True, False), (False, True)])
def test_products_equal_scipy(degree, masked, empty):
    import torch
    from waterscapes_amd import amg, levels as lv
    A = _laplacian(5, 0.1)
    n = A.shape[0]
    mask = np.zeros(n, dtype=bool)
    if masked:
        mask[::6] = True
        free = sp.diags((~mask).astype(float))
        A = (free @ A @ free + sp.diags(mask.astype(float))).tocsr()
        A.sort_indices()
    lev = amg.setup_host(A.indptr, A.indices, A.data, amg.AmgParams(max_coarse=5))[0][0]
    P = sp.csr_matrix((lev["P_v"], lev["P_ci"], lev["P_rp"]), shape=(n, lev["nc"]))
    dinv = lev["dinv"].copy()
    if empty:                                # a padded level: no matrix, P = I
        A = sp.csr_matrix((n, n))
        P = sp.identity(n, format="csr")
        dinv[:] = 0.0
    R = P.T.tocsr()
    R.sort_indices()

    def dev(M):
        return (torch.as_tensor(M.indptr.astype(np.int32)),
                torch.as_tensor(M.indices.astype(np.int32)), torch.as_tensor(M.data))
    c0 = 0.7
    f = lv.fused_transfers(dev(A), dev(P), dev(R), torch.as_tensor(dinv), degree, c0,
                           torch.as_tensor(mask) if masked else None, values=_host_values)
    live = sp.diags((~mask).astype(float))
    AP, RA = live @ (A @ P), (R @ A) @ live
    nc = P.shape[1]

    def csr(rp, ci, v, shape):
        return sp.csr_matrix((v, f[ci].numpy(), f[rp].numpy()), shape=shape).toarray()
    if degree == 1:
        W = csr("W_rp", "W_ci", f["W_v"].numpy(), (nc, n))
        Q = csr("Q_rp", "Q_ci", f["Q_v"].numpy(), (n, nc))
        assert np.abs(W - ((R @ live) - c0 * RA @ sp.diags(dinv)).toarray()).max() <= 1e-13
        assert np.abs(Q - (live @ P - c0 * sp.diags(dinv) @ AP).toarray()).max() <= 1e-13
    else:
        W = csr("W_rp", "W_ci", f["W_v"].numpy(), (nc, 2 * n))
        assert np.abs(W - np.hstack([-RA.toarray(), (R @ live).toarray()])).max() <= 1e-13
        q = f["Q_v"].numpy().reshape(-1, 2)
        assert np.abs(csr("Q_rp", "Q_ci", q[:, 0], (n, nc)) - AP.toarray()).max() <= 1e-13
        assert np.abs(csr("Q_rp", "Q_ci", q[:, 1], (n, nc)) - (live @ P).toarray()).max() <= 1e-13


@pytest.mark.parametrize("degree", [1, 2])
@pytest.mark.parametrize("choice", [(True, False), (False, True), (False, False)])
def test_only_the_chosen_products_are_formed(degree, choice, monkeypatch):
    """The choice is made from the sizes the products would have; the other
    product's values are not formed, and a sliced Q replaces its CSR form."""
    import torch
    from waterscapes_amd import amg, levels as lv
    A = _laplacian(5, 0.1)
    lev = amg.setup_host(A.indptr, A.indices, A.data, amg.AmgParams(max_coarse=5))[0][0]
    formed = []

    def values(*a):
        formed.append(a[0].numel())
        return _host_values(*a)

    def csr(k):
        return tuple(torch.as_tensor(lev[k + e]).to(torch.float64 if e == "_v" else torch.int32)
                     for e in ("_rp", "_ci", "_v"))
    args = csr("A"), csr("P"), csr("R"), torch.as_tensor(lev["dinv"]), degree, 0.7
    full = lv.fused_transfers(*args, values=values)
    formed.clear()
    sizes = {}
    got = lv.fused_transfers(*args, values=values,
                             use=lambda f: sizes.update((k, v.numel()) for k, v in f.items())
                             or choice)
    assert sizes == {k: full[k].numel() for k in ("W_ci", "Q_ci", "Q_v")}
    assert len(formed) == sum(choice)
    assert set(got) == {k for k in full if choice["WQ".index(k[0])]}
    assert all(torch.equal(got[k], full[k]) for k in got)
    ld = dict(got, A_rp=args[0][0], A_ci=args[0][1], A_v=args[0][2])
    monkeypatch.setattr(lv, "SLICE_ROWS", 1)
    lv.add_slices(ld, lev["n"])
    assert ("Q_s" in ld) == ("Q_v" in ld) == choice[1] and "Q_ci" not in ld
    if choice[1]:
        assert ld["Q_v"] is ld["Q_s"]["v"]


@pytest.mark.parametrize("n,m,density", [(1, 5, 0.0), (64, 64, 0.05), (65, 3, 1.0),
                                         (1000, 400, 0.02), (1537, 65536, 0.01)])
@pytest.mark.parametrize("pair", [False, True])
def test_slices_hold_the_matrix(n, m, density, pair):
    import torch
    from waterscapes_amd import levels as lv
    M = sp.random(n, m, density, random_state=1, format="csr")
    M.sort_indices()
    v = torch.as_tensor(np.stack([M.data, 2 * M.data], 1) if pair else M.data)
    s = lv.slices(torch.as_tensor(M.indptr), torch.as_tensor(M.indices), v, n)
    off, base, row, val = (s[k].numpy() for k in ("off", "base", "row", "v"))
    dc = lv._u16(s["dc"]).numpy().view(np.uint16)
    assert len(off) == len(base) + 1 == (n + 63) // 64 + 1 and len(row) == 64 * len(base)
    assert np.array_equal(np.sort(row[row >= 0]), np.arange(n))
    assert len(val) == len(dc) == 64 * off[-1]
    got = np.zeros((n, m))
    for at in np.flatnonzero(row >= 0):
        sl = at // 64
        k = 64 * (off[sl] + np.arange(off[sl + 1] - off[sl])) + at % 64
        assert len(k) == 0 or (base[sl] + dc[k]).max() < m
        x = val[k, 1] / 2 if pair else val[k]
        np.add.at(got[row[at]], base[sl] + dc[k], x)
    assert np.array_equal(got, M.toarray())


@pytest.mark.parametrize("sizes", [(700, 900), (64, 1, 513), (27, 30, 5, 700)])
@pytest.mark.parametrize("broken", [0, 1])
def test_slices_stay_inside_an_instance(sizes, broken):
    """Rows of a packed level's other instances do not read an instance whose
    vector is NaN, padding entries and rows without entries included; each
    row's sum is its matrix row's."""
    import torch
    from waterscapes_amd import levels as lv
    blocks = [sp.random(k, k, 0.02, random_state=i, format="lil") for i, k in enumerate(sizes)]
    for b in blocks:
        b[b.shape[0] // 2] = 0.0                     # a row without entries
    blocks[-1][:] = 0.0                              # a padded level: no matrix
    blocks[-2][::3, :] = 1.0                         # padding beside long rows
    M = sp.block_diag(blocks, format="csr")
    M.eliminate_zeros()
    M.sort_indices()
    n = M.shape[0]
    grp = np.repeat(np.arange(len(sizes), dtype=np.int32), sizes)
    s = lv.slices(torch.as_tensor(M.indptr), torch.as_tensor(M.indices),
                  torch.as_tensor(M.data), n, torch.as_tensor(grp))
    off, base, row, dc, v = (s[k].numpy() for k in ("off", "base", "row", "dc", "v"))
    assert np.array_equal(np.sort(row[row >= 0]), np.arange(n))
    x = np.random.default_rng(0).standard_normal(n)
    ref = M @ x
    x[grp == broken] = np.nan
    y = np.full(n, np.nan)
    for at in np.flatnonzero(row >= 0):              # as sell_part: padding multiplies too
        k = 64 * np.arange(off[at // 64], off[at // 64 + 1]) + at % 64
        y[row[at]] = (v[k] * x[base[at // 64] + dc[k]]).sum()
    others = grp != broken
    assert not np.isnan(y[others]).any()
    assert np.abs(y[others] - ref[others]).max() <= 1e-13 * np.abs(ref).max()
    assert len(base) == sum((k + 63) // 64 for k in sizes) == len(off) - 1


def test_slices_refuse_wide_columns():
    import torch
    from waterscapes_amd import levels as lv
    rp, ci = torch.tensor([0, 2]), torch.tensor([0, 1 << 16])
    assert lv.slices(rp, ci, torch.ones(2), 1) is None
    assert lv.slices(rp, ci - torch.tensor([0, 1]), torch.ones(2), 1) is not None


@pytest.mark.gpu
@pytest.mark.parametrize("slice_rows,mixed_choice", [(1 << 30, False), (1 << 30, True),
                                                     (600, True), (1, False), (1, True)])
@pytest.mark.parametrize("n,A,degs", [(3, 1, (1,)), (5, 3, (1,)), (5, 2, (2,)), (6, 6, (3, 1)),
                                      (27, 1, (1,)), (27, 1, (2,))])
@pytest.mark.parametrize("mode", ["fp64", "mixed"])
def test_preconditioner_with_fused_transfers(n, A, degs, mode, slice_rows, mixed_choice,
                                              monkeypatch):
    import torch
    from test_gpu_solver import _ref_precond, _setup
    from waterscapes_amd import levels as lv
    from waterscapes_amd.amg import AmgParams
    monkeypatch.setattr(lv, "DENSE_TAIL_BYTES", 30 * 30 * 8)
    monkeypatch.setattr(lv, "SLICE_ROWS", slice_rows)
    # every combination of the two fused transfers, level by level
    turn = iter([(True, True), (False, True), (True, False), (False, False)] * 8)
    monkeypatch.setattr(lv, "worth_fusing",
                        lambda *a: next(turn) if mixed_choice else (True, True))
    big = dict(max_coarse=25) if n < 20 else {}
    _, _, dev, solver, dofs, _ = _setup(
        n=n, A=A, mode=mode, compact_plevel0=False, autotune=False,
        amg=AmgParams(smoother_degree=3, level_degrees=degs, **big), pamg=AmgParams(**big))
    assert len(solver.levels) >= 3 and len(solver.plevels) >= 2
    dev_levels = solver._level_arrays(0 if mode == "fp64" else 1)
    for (levs, _), host in zip(dev_levels, (solver.levels, solver.plevels)):
        for ld, lev in zip(levs[:-1], host):
            assert ("A_s" in ld) == (lev["n"] >= slice_rows)
            assert mixed_choice or ("W_v" in ld and "Q_v" in ld)
    r = np.random.default_rng(2).standard_normal(dev.n)
    r[np.concatenate(dofs)] = 0.0
    dtype = torch.float64 if mode == "fp64" else torch.float32
    x = torch.tensor(r, device="cuda", dtype=dtype)
    z = solver.precond(x, 0 if mode == "fp64" else 1).double().cpu().numpy()
    again = solver.precond(x, 0 if mode == "fp64" else 1).double().cpu().numpy()
    assert np.array_equal(z, again)
    ref = _ref_precond(solver, r, compact=mode == "mixed")
    tol = 1e-12 if mode == "fp64" else 1e-5
    nu = dev.nu
    for a, b in ((z[:nu], ref[:nu]), (z[nu:], ref[nu:])):
        assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b)
    solver.close()


def test_worth_fusing_by_bytes():
    """W while it reads less than a launch's bytes more than R, Q while less
    than a launch's bytes more than P and the level operator."""
    import torch
    from waterscapes_amd import levels as lv

    def ld(nnz, compact=False):
        d = dict(A_ci=torch.zeros(nnz), P_ci=torch.zeros(1000))
        return dict(d, A_v16=None) if compact else d

    def f(w, q, pair):
        return dict(W_ci=torch.zeros(w), Q_ci=torch.zeros(q), Q_v=torch.zeros(q * (1 + pair)))
    launch = int(lv.LAUNCH_BYTES)
    assert lv.worth_fusing(ld(10**4), f(10**4, 10**4, 1), 4, 1000) == (True, True)
    w = launch // 8 + 1000                    # 8 bytes an entry in FP32
    assert lv.worth_fusing(ld(10**4), f(w - 1, 10, 0), 4, 1000)[0]
    assert not lv.worth_fusing(ld(10**4), f(w + 1, 10, 0), 4, 1000)[0]
    q = (launch + 8 * 1000 + 4 * 10**6) // 8
    assert lv.worth_fusing(ld(10**6, True), f(10, q - 1, 0), 4, 1000)[1]
    assert not lv.worth_fusing(ld(10**6, True), f(10, q + 1, 0), 4, 1000)[1]
