"""Derived operators of an AMG hierarchy, made once per solver on the device.

Dense tail: a V-cycle is a fixed linear operator, so the part of it below
some level is one dense matrix M of that level's size.  Where M is small
enough, applying it (one launch) replaces the smoothing, residual, transfer
and coarse-solve launches of that level and every coarser one (four to nine
dependent launches per level, each a few microseconds whatever its size).
M is formed in FP64 from the same level values the V-cycle kernels read.
The reference leaves the cycle to hypre
(mpet/mpettotalpressuresolver.py:448).
"""
from __future__ import annotations

import torch

from .amg import chebyshev_coefficients

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


def tail_start(levels, rows):
    """The finest level of at most `rows` rows (the coarsest if none is)."""
    for l, lev in enumerate(levels):
        if lev["n"] <= rows:
            return l
    return len(levels) - 1


def with_dense_tail(levels, cinv, rows, params, device, values=None, mask0=None, first=0):
    """(levels, cinv) of the hierarchy cut at its finest level of at most
    `rows` rows (not before level `first`), whose coarsest operator (device
    FP64 tensor) is the V-cycle that began there."""
    start = max(tail_start(levels, rows), min(first, len(levels) - 1))
    if start == len(levels) - 1:
        return levels, cinv
    M = dense_tail(levels, cinv, start, params, device, values, mask0)
    last = dict(levels[start], nc=0)
    for k in ("P_rp", "P_ci", "P_v", "R_rp", "R_ci", "R_v"):
        last.pop(k, None)
    return list(levels[:start]) + [last], M
