"""Derived operators of an AMG hierarchy, made once per solver on the device.

Dense tail: a V-cycle is a fixed linear operator, so the part of it below
some level is one dense matrix M of that level's size.  Where M is small
enough, applying it (one launch) replaces the smoothing, residual, transfer
and coarse-solve launches of that level and every coarser one (four to nine
dependent launches per level, each a few microseconds whatever its size).
M is formed in FP64 from the same level values the V-cycle kernels read.

Fused transfers: on the levels that stay sparse, residual and restriction
are one launch with W and prolongation and the first post-smoothing step
one with Q (csrc/amg_cycle.h, "Fused transfers"), formed here from R A and
A P, where their bytes do not cost more than the launch they save.

The reference leaves the cycle to hypre
(mpet/mpettotalpressuresolver.py:448).
"""
from __future__ import annotations

import ctypes as C

import torch

from . import _lib
from ._lib import check, ptr
from .amg import chebyshev_coefficients

class Slices(C.Structure):
    _fields_ = [("off", C.c_void_p), ("base", C.c_void_p), ("row", C.c_void_p),
                ("dc", C.c_void_p), ("count", C.c_int32)]


# A dense tail is used up to this many bytes of M.  Streaming it costs bytes
# / ~4.5 TB/s (64 MiB: 15 us) against about four launches per replaced level
# at 4-5 us each.
DENSE_TAIL_BYTES = 64 << 20


def dense_rows(size, bytes_=None):
    """Most rows of a dense tail with values of `size` bytes."""
    return int((DENSE_TAIL_BYTES if bytes_ is None else bytes_) ** 0.5 / size ** 0.5)


def host_array(m):
    """A coarsest operator (host array or device tensor) as a host array."""
    return m.cpu().numpy() if torch.is_tensor(m) else m


def _dense(rp, ci, v, n, m, dev):
    rp = torch.as_tensor(rp).to(dev).long()
    ci = torch.as_tensor(ci).to(dev).long()
    v = torch.as_tensor(v).to(dev, torch.float64)
    rows = torch.repeat_interleave(torch.arange(n, device=dev), rp[1:] - rp[:-1])
    out = torch.zeros(n, m, dtype=torch.float64, device=dev)
    out[rows, ci] = v
    return out


def dense_tail(levels, cinv, start, params, device, values=None, mask0=None):
    """The V-cycle of levels[start:] (dense inverse cinv on the coarsest) as
    a dense FP64 matrix on `device`.  values(l): the level-l operator (rp, ci,
    v) to use instead of the level's own (None: the level's own); mask0:
    level-0 rows held at zero."""
    M = torch.as_tensor(cinv).to(device, torch.float64)
    for l in range(len(levels) - 2, start - 1, -1):
        lev = levels[l]
        n, nc = lev["n"], lev["nc"]
        a = values(l) if values is not None else None
        A = _dense(*(a or (lev["A_rp"], lev["A_ci"], lev["A_v"])), n, n, device)
        P = _dense(lev["P_rp"], lev["P_ci"], lev["P_v"], n, nc, device)
        D = torch.as_tensor(lev["dinv"]).to(device, torch.float64)[:, None].clone()
        keep = None
        if l == 0 and mask0 is not None:
            keep = (~mask0.to(device).bool()).to(torch.float64)[:, None]
            D *= keep
        deg = params.degree(l)
        lmax = lev["rho"] * params.eig_safety
        cd, cr = (c.tolist() for c in chebyshev_coefficients(lmax / params.eig_ratio, lmax, deg))

        def residual(X):                       # I - A X
            R = torch.matmul(A, X).neg_()
            R.diagonal().add_(1.0)
            return R
        d = torch.diag(cr[0] * D[:, 0])
        X = d.clone()
        for i in range(1, deg):
            d = cd[i] * d + residual(X).mul_(cr[i] * D)
            X += d
        R = residual(X)
        if keep is not None:
            R *= keep
        X += torch.matmul(P, torch.matmul(M, torch.matmul(P.t(), R)))
        if keep is not None:
            X *= keep
        for i in range(deg):
            step = residual(X).mul_(cr[i] * D)
            d = step if i == 0 else step + cd[i] * d
            X += d
        M = X
    return M


def column_ranges(M):
    """(n, 4) int32: two column runs [c0, c1), [c2, c3) of every row of M that
    hold its nonzeros: the first to the last nonzero without the row's
    longest inner run of zeros (empty runs for a zero row)."""
    n = M.shape[1]
    j = torch.arange(n, dtype=torch.int32, device=M.device)
    nz = M != 0
    last = torch.where(nz, j, -1).cummax(dim=1).values      # last nonzero up to j
    prev = torch.nn.functional.pad(last[:, :-1], (1, 0), value=-1)
    gap, c2 = torch.where(nz & (prev >= 0), j - prev - 1, 0).max(dim=1)
    c0 = torch.where(nz, j, n).amin(dim=1)
    c3 = last[:, -1] + 1
    c2 = torch.where(gap > 0, c2.to(torch.int32), c3)
    some = nz.any(dim=1)
    out = torch.stack([c0, c2 - gap, c2, c3], dim=1) * some[:, None]
    return out.to(torch.int32).contiguous()


def tail_start(levels, rows, first=0):
    """The finest level of at most `rows` rows, not before level `first` (the
    coarsest if none is)."""
    for l, lev in enumerate(levels):
        if l >= first and lev["n"] <= rows:
            return l
    return len(levels) - 1


def with_dense_tail(levels, cinv, rows, params, device, values=None, mask0=None, first=0):
    """(levels, cinv) of the hierarchy cut at tail_start(levels, rows, first),
    whose coarsest operator (device FP64 tensor) is the V-cycle that began
    there."""
    start = tail_start(levels, rows, first)
    if start == len(levels) - 1:
        return levels, cinv
    M = dense_tail(levels, cinv, start, params, device, values, mask0)
    last = dict(levels[start], nc=0)
    for k in ("P_rp", "P_ci", "P_v", "R_rp", "R_ci", "R_v"):
        last.pop(k, None)
    return list(levels[:start]) + [last], M


# ---------------------------------------------------------------------------
# fused transfers
# ---------------------------------------------------------------------------
# products (A row entry, P row entry) expanded at a time: bounds the sort's
# memory to ~1 GB
_CHUNK = 1 << 25


def _product_keys(A, P, nc):
    """Sorted unique keys row * nc + column of the patterns of A P and P."""
    (arp, aci), (prp, pci) = A, P
    dev = aci.device
    arp, prp = arp.long(), prp.long()
    n = arp.numel() - 1
    plen = prp[1:] - prp[:-1]
    per_nz = plen[aci.long()]                            # products of each A entry
    ends = torch.cumsum(per_nz, 0) if per_nz.numel() else per_nz
    total = int(ends[-1]) if ends.numel() else 0
    rows = torch.repeat_interleave(torch.arange(n, device=dev), arp[1:] - arp[:-1])
    prow = torch.repeat_interleave(torch.arange(n, device=dev), plen)
    keys = [prow * nc + pci.long()]                      # rows of A may be empty
    at, done = 0, 0
    while done < total:
        # whole A entries up to about _CHUNK products
        stop = int(torch.searchsorted(ends, min(done + _CHUNK, total), right=False)) + 1
        cnt = per_nz[at:stop]
        rep = torch.repeat_interleave(torch.arange(at, stop, device=dev), cnt)
        first = ends[at:stop] - cnt
        off = torch.arange(done, done + rep.numel(), device=dev) - first[rep - at]
        cols = pci[prp[aci[rep].long()] + off].long()
        keys.append(torch.unique(rows[rep] * nc + cols))
        done += rep.numel()
        at = stop
    return torch.unique(torch.cat(keys))


def _row_pointers(rows, n):
    out = torch.zeros(n + 1, dtype=torch.int64, device=rows.device)
    out[1:] = torch.cumsum(torch.bincount(rows, minlength=n), 0)
    return out


def _csr(rows, n, cols, what):
    rp = _row_pointers(rows, n)
    if int(rp[-1]) >= 2**31:
        raise ValueError(f"{what}: too large for 32-bit row pointers")
    return rp.to(torch.int32), cols.to(torch.int32)


def _values(rows, cols, X, Y):
    out = torch.empty(rows.numel(), dtype=torch.float64, device=rows.device)
    r, c = rows.to(torch.int32), cols.to(torch.int32)
    check(_lib.lib().mpet_product_values(r.numel(), ptr(r), ptr(c), *(ptr(t) for t in X),
                                         *(ptr(t) for t in Y), ptr(out), _lib.stream_ptr()))
    return out


def fused_transfers(A, P, R, dinv, degree, c0, mask=None, values=_values, use=None):
    """W and Q of one level from its device matrices A, P, R = (rp, ci, FP64
    values) with sorted int32 columns: dict of W_rp, W_ci, W_v, Q_rp, Q_ci,
    Q_v (FP64 values; Q_v holds pairs for degree > 1).  dinv: FP64 diagonal
    inverse, c0: the first Chebyshev coefficient, mask: rows held at zero.
    use(f): (form W, form Q) from their sizes alone, f a dict of W_ci, Q_ci and
    Q_v without storage (None: both)."""
    n, nc = A[0].numel() - 1, R[0].numel() - 1
    key = _product_keys(A[:2], P[:2], max(nc, 1))
    use_w = use_q = True
    if use is not None:
        nnz, many = key.numel(), degree > 1
        use_w, use_q = use({k: torch.empty(m, device="meta") for k, m in
                            (("W_ci", nnz + (R[1].numel() if many else 0)), ("Q_ci", nnz),
                             ("Q_v", nnz * (1 + many)))})
    dead = None if mask is None else mask.bool()
    out = {}
    if use_q:
        out.update(_fused_prolongation(A, P, dinv, degree, c0, dead, key, n, nc, values))
    if use_w:
        out.update(_fused_restriction(A, R, dinv, degree, c0, dead, key, n, nc, values))
    return out


def _fused_prolongation(A, P, dinv, degree, c0, dead, key, n, nc, values):
    """A P and P on the pattern of A P."""
    rows, cols = key // nc, key % nc
    ap = values(rows, cols, A, P)
    prow = torch.repeat_interleave(torch.arange(n, device=key.device),
                                   (P[0][1:] - P[0][:-1]).long())
    p = torch.zeros_like(ap)
    p[torch.searchsorted(key, prow * nc + P[1].long())] = P[2]
    if dead is not None:
        ap[dead[rows]] = 0.0
        p[dead[rows]] = 0.0
    q = p - c0 * dinv[rows] * ap if degree == 1 else torch.stack([ap, p], 1).reshape(-1)
    q_rp, q_ci = _csr(rows, n, cols, "fused prolongation")
    return dict(Q_rp=q_rp, Q_ci=q_ci, Q_v=q)


def _fused_restriction(A, R, dinv, degree, c0, dead, key, n, nc, values):
    """R A on the transposed pattern of A P, with R."""
    rows, cols = key // nc, key % nc
    order = torch.argsort(cols * n + rows)
    wr, wc = cols[order], rows[order]
    ra = values(wr, wc, R, A)
    rrow = torch.repeat_interleave(torch.arange(nc, device=key.device),
                                   (R[0][1:] - R[0][:-1]).long())
    rcol, rv = R[1].long(), R[2].clone()
    if dead is not None:
        ra[dead[wc]] = 0.0
        rv[dead[rcol]] = 0.0
    if degree == 1:
        w = -c0 * dinv[wc] * ra
        w[torch.searchsorted(wr * n + wc, rrow * n + rcol)] += rv
    else:
        # row-wise [-R A, R], the columns of R shifted by n
        ra_rp, r_rp = _row_pointers(wr, nc), R[0].long()
        at_ra = torch.arange(wr.numel(), device=key.device) + r_rp[wr]
        at_r = torch.arange(rrow.numel(), device=key.device) + ra_rp[rrow + 1]
        total = wr.numel() + rrow.numel()
        w = torch.empty(total, dtype=torch.float64, device=key.device)
        col = torch.empty(total, dtype=torch.int64, device=key.device)
        row = torch.empty(total, dtype=torch.int64, device=key.device)
        w[at_ra], w[at_r] = -ra, rv
        col[at_ra], col[at_r] = wc, rcol + n
        row[at_ra], row[at_r] = wr, rrow
        wr, wc = row, col
    w_rp, w_ci = _csr(wr, nc, wc, "fused restriction")
    return dict(W_rp=w_rp, W_ci=w_ci, W_v=w)


# ---------------------------------------------------------------------------
# sliced rows
# ---------------------------------------------------------------------------
# Levels of at least this many rows run one thread per row on sliced copies:
# 65,536 rows are 1,024 waves, four per compute unit; below, several lanes
# share a row.  The line also decides between the two branches of a captured
# graph (a sliced level) and joint launches of both V-cycles (none, amg_cycle.h
# joint_ok), and lies where neither wins clearly.  An iteration sliced and forked
# / not sliced, us: direct A = 2 at 16^3 (35,937 P2 rows) 115 / 106, 18^3 126 /
# 124, 20^3 (68,921) 122 / 122, 22^3 132 / 132; mixed A = 4 at 16^3 100 / 101,
# 20^3 106 / 110, 22^3 134 / 122, 24^3 140 / 134, 28^3 157 / 149 (forked either
# way there); mixed A = 1 at 16^3 93 / 88, 20^3 104 / 97, 24^3 116 / 116, 28^3
# (185,193) 133 / 140; at 48^3 (912,673) joint launches cost 474, slices 425.
SLICE_ROWS = 1 << 16
# rows are sorted by length within windows of this many (a multiple of 64)
WINDOW = 512


def slices(rp, ci, values, n, grp=None):
    """Sliced copy (include/mpet_hip.h, MpetSlices) of a CSR matrix with n
    rows on its device: dict of off, base, row, dc and v (values: (nnz,) or
    (nnz, 2)), or None where the columns of some slice span 2^16 or more.

    grp: the instance of each row of a packed level, not decreasing.  Windows
    and slices hold rows of one instance only: a padding entry multiplies a
    column of its slice by zero, and 0 x NaN from an instance that broke down
    must not reach another one's rows."""
    dev = ci.device
    rp, ci = rp.long(), ci.long()
    length = rp[1:] - rp[:-1]
    at = torch.arange(n, device=dev)
    grp = torch.zeros_like(at) if grp is None else grp.to(dev).long()
    rows = torch.bincount(grp) if n else at              # of each instance
    mine = at - (torch.cumsum(rows, 0) - rows)[grp]      # row within the instance

    def chunks(size):                    # of an instance's rows, and its first
        cnt = (rows + size - 1) // size
        return int(cnt.sum()), (torch.cumsum(cnt, 0) - cnt)[grp]
    ns, first_slice = chunks(64)
    _, first_window = chunks(WINDOW)
    longest = int(length.max()) + 1 if n else 1
    order = torch.argsort((first_window + mine // WINDOW) * longest + (longest - 1 - length),
                          stable=True)
    # instances stay in place, so sorted position i is of instance grp[i]
    place = torch.empty(n, dtype=torch.int64, device=dev)
    place[order] = 64 * first_slice + mine               # slot of each row
    row = torch.full((64 * ns,), -1, dtype=torch.int64, device=dev)
    row[place] = at
    width = torch.zeros(64 * ns, dtype=torch.int64, device=dev)
    width[place] = length
    width = width.view(ns, 64).amax(1)
    off = torch.zeros(ns + 1, dtype=torch.int64, device=dev)
    off[1:] = torch.cumsum(width, 0)
    total = 64 * int(off[-1])
    of = torch.repeat_interleave(at, length)             # row of each entry
    slot = place[of]
    j = torch.arange(ci.numel(), device=dev) - rp[of]
    dest = (off[slot // 64] + j) * 64 + slot % 64
    base = torch.full((ns,), 2**31 - 1, dtype=torch.int64, device=dev)
    base.scatter_reduce_(0, slot // 64, ci, "amin")
    base[width == 0] = 0
    delta = ci - base[slot // 64]
    if total >= 2**37 or (delta.numel() and int(delta.max()) >= 1 << 16):
        return None
    dc = torch.zeros(total, dtype=torch.int32, device=dev)
    dc[dest] = delta.to(torch.int32)
    v = torch.zeros((total,) + tuple(values.shape[1:]), dtype=values.dtype, device=dev)
    v[dest] = values
    return dict(off=off.to(torch.int32), base=base.to(torch.int32), row=row.to(torch.int32),
                dc=dc, v=v)


def _u16(dc):
    """int32 offsets below 2^16 as 16-bit words (the bits of uint16)."""
    return torch.where(dc >= 1 << 15, dc - (1 << 16), dc).to(torch.int16)


def add_slices(ld, n):
    """Sliced copies of a level operator and of its Q, where one thread per
    row fills the chip."""
    if n < SLICE_ROWS:
        return
    grp = ld.get("grp")
    if "A_v16" in ld:
        s = slices(ld["A_rp"], ld["A_ci"], ld["A_v16"], n, grp)
        if s is not None:            # half | offset << 16 in one 32-bit word
            bits = s["v"].view(torch.int16).to(torch.int32) & 0xffff
            word = bits | (_u16(s["dc"]).to(torch.int32) << 16)
            ld["A_s"] = dict(s, v=word, dc=None)
    else:
        s = slices(ld["A_rp"], ld["A_ci"], ld["A_v"], n, grp)
        if s is not None:
            ld["A_s"] = dict(s, dc=_u16(s["dc"]))
    if "Q_v" in ld:
        q = ld["Q_v"].view(ld["Q_ci"].numel(), -1)
        s = slices(ld["Q_rp"], ld["Q_ci"], q, n, grp)
        if s is not None:            # instead of the CSR form
            ld["Q_s"] = dict(s, dc=_u16(s["dc"]))
            ld["Q_v"] = s["v"]
            del ld["Q_rp"], ld["Q_ci"]


def _describe_slices(S, s):
    S.off, S.base, S.row, S.dc = (ptr(s[k]) for k in ("off", "base", "row", "dc"))
    S.count = s["base"].numel()


def add_fused(levs, hosts, params, dtype, mask0=None):
    """Fused transfers of every level but the coarsest that is worth it, and
    sliced copies, added to the uploaded level dicts `levs` (values in their
    precision); hosts: the host levels (rho)."""
    for l, ld in enumerate(levs[:-1]):
        if "A_v16" in ld:
            av = ld["A_v16"].double() * ld["vscale"]
        else:
            av = ld["A_v"].double()
        deg = params.degree(l)
        lmax = hosts[l]["rho"] * params.eig_safety
        c0 = float(chebyshev_coefficients(lmax / params.eig_ratio, lmax, deg)[1][0])
        size, n = (8 if dtype == 0 else 4), int(hosts[l]["n"])
        f = fused_transfers((ld["A_rp"], ld["A_ci"], av),
                            (ld["P_rp"], ld["P_ci"], ld["P_v"].double()),
                            (ld["R_rp"], ld["R_ci"], ld["R_v"].double()), ld["dinv"].double(),
                            deg, c0, mask0 if l == 0 else None,
                            use=lambda f, ld=ld, n=n: worth_fusing(ld, f, size, n))
        tdt = torch.float64 if dtype == 0 else torch.float32
        ld.update({k: v.to(tdt) if k in ("W_v", "Q_v") else v for k, v in f.items()})
        add_slices(ld, n)


# Bytes that take as long as the launch a fused transfer saves: about 3 us of
# a kernel that streams at 4.5 TB/s.
LAUNCH_BYTES = 13.5e6


def worth_fusing(ld, f, size, n):
    """(use W, use Q) of a level: W is read instead of R, in one launch with
    the residual instead of after it; Q instead of P and the level operator."""
    def matrix(nnz, value):
        return nnz * (value + 4)
    a = ld["A_ci"].numel() * (4 if "A_v16" in ld else (size + 2 if n >= SLICE_ROWS
                                                       else size + 4))
    pr = matrix(ld["P_ci"].numel(), size)
    w = matrix(f["W_ci"].numel(), size)
    q = f["Q_v"].numel() * size + f["Q_ci"].numel() * (2 if n >= SLICE_ROWS else 4)
    return w < pr + LAUNCH_BYTES, q < pr + a + LAUNCH_BYTES


def _log2_lanes(avg, rows, nc):
    """Lanes per row of W and Q (log2): about eight nonzeros a lane, more
    while the launch would hold fewer than 2^19 lanes; three columns need at
    least four lanes."""
    lg = 2 if nc == 3 else 0
    while (8 << lg) < avg and lg < 6:
        lg += 1
    while (rows << lg) < (1 << 19) and (1 << lg) < avg and lg < 6:
        lg += 1
    return lg


def describe_fused(L, ld, n, ncoarse, nc):
    """Fill the fused-transfer part of an AmgLevelDesc."""
    if "W_v" in ld:
        L.W_rp, L.W_ci, L.W_v = ptr(ld["W_rp"]), ptr(ld["W_ci"]), ptr(ld["W_v"])
        L.lgW = _log2_lanes(ld["W_ci"].numel() / max(ncoarse, 1), ncoarse, nc)
    if "Q_v" in ld:
        L.Q_v = ptr(ld["Q_v"])
        if "Q_ci" in ld:
            L.Q_rp, L.Q_ci = ptr(ld["Q_rp"]), ptr(ld["Q_ci"])
            L.lgQ = _log2_lanes(ld["Q_ci"].numel() / max(n, 1), n, nc)
    if "A_s" in ld:
        _describe_slices(L.A_s, ld["A_s"])
        L.A_sv = ptr(ld["A_s"]["v"])
    if "Q_s" in ld:
        _describe_slices(L.Q_s, ld["Q_s"])
