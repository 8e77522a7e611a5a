"""Host smoothed-aggregation setup (csrc/amg_setup.cpp) on the CPU: the
dense inverse of the coarsest operator is the inverse (A_c Cinv = I,
symmetric) and does not depend on the OpenMP thread count; the levels are
Galerkin products R A P with R = P^T."""
import os
import subprocess
import sys

import numpy as np
import pytest
import scipy.sparse as sp

from waterscapes_amd import amg


def _lap3d(n):
    """7-point Laplacian on an n^3 grid plus a small shift (SPD)."""
    e = np.ones(n)
    T = sp.diags([-e[:-1], 2 * e, -e[:-1]], [-1, 0, 1])
    I = sp.identity(n)
    A = sp.kron(sp.kron(T, I), I) + sp.kron(sp.kron(I, T), I) + sp.kron(sp.kron(I, I), T)
    return (A + 1e-3 * sp.identity(n ** 3)).tocsr()


def test_coarse_inverse_and_galerkin_levels():
    A = _lap3d(14)
    A.sort_indices()
    levels, cinv = amg.setup_host(A.indptr, A.indices, A.data,
                                  amg.AmgParams(max_coarse=700, max_levels=8))
    assert len(levels) >= 2
    last = levels[-1]
    Ac = sp.csr_matrix((last["A_v"], last["A_ci"], last["A_rp"]), shape=(last["n"],) * 2)
    I = Ac.toarray() @ cinv
    assert np.abs(I - np.eye(last["n"])).max() <= 1e-10
    assert np.array_equal(cinv, cinv.T)
    for l in range(len(levels) - 1):
        lev, nxt = levels[l], levels[l + 1]
        Al = sp.csr_matrix((lev["A_v"], lev["A_ci"], lev["A_rp"]), shape=(lev["n"],) * 2)
        P = sp.csr_matrix((lev["P_v"], lev["P_ci"], lev["P_rp"]), shape=(lev["n"], lev["nc"]))
        An = sp.csr_matrix((nxt["A_v"], nxt["A_ci"], nxt["A_rp"]), shape=(nxt["n"],) * 2)
        G = (P.T @ Al @ P).toarray()
        assert np.abs(G - An.toarray()).max() <= 1e-12 * np.abs(G).max()


def test_coarse_inverse_independent_of_thread_count():
    code = ("import numpy as np, scipy.sparse as sp, sys; sys.path.insert(0, %r);"
            "from tests.test_amg_setup import _lap3d; from waterscapes_amd import amg;"
            "A = _lap3d(12); A.sort_indices();"
            "lv, ci = amg.setup_host(A.indptr, A.indices, A.data, amg.AmgParams(max_coarse=900));"
            "sys.stdout.buffer.write(ci.tobytes())") % os.path.dirname(os.path.dirname(
                os.path.abspath(__file__)))
    outs = []
    for t in ("1", "4"):
        env = dict(os.environ, OMP_NUM_THREADS=t)
        outs.append(subprocess.run([sys.executable, "-c", code], env=env, check=True,
                                   capture_output=True).stdout)
    assert len(outs[0]) > 0 and outs[0] == outs[1]


@pytest.mark.parametrize("tensors", [False, True])
def test_compact_level(tensors):
    """Half values and 16-bit offsets of a level operator, from a pattern of
    host arrays or tensors; refused where an offset or a diagonal is out of
    range."""
    import torch
    from waterscapes_amd.krylov import compact_level
    n = 40000
    rp = np.arange(0, 2 * n + 1, 2, dtype=np.int64)
    ci = np.stack([np.maximum(np.arange(n) - 32767, 0), np.arange(n)], 1).astype(np.int32)
    ci[0] = 0, 5
    v = torch.as_tensor(np.random.default_rng(0).uniform(0.1, 3.0, 2 * n))

    def pattern(c):
        return (torch.as_tensor(rp.astype(np.int32)), torch.as_tensor(c)) if tensors else (rp, c)
    c = compact_level(pattern(ci.reshape(-1)), v, 2.0 ** -22)
    rows = np.repeat(np.arange(n), 2)
    assert np.array_equal(c["A_dci"].numpy().astype(np.int64) + rows, ci.reshape(-1))
    assert c["A_dci"].dtype == torch.int16 and c["A_v16"].dtype == torch.float16
    assert 2.0 ** 9 <= float(c["A_v16"].max()) <= 2.0 ** 10
    assert torch.equal(c["A_v16"], (v / c["vscale"]).half())
    tiny = v.clone()
    tiny[2 * 7 + 1] = 1e-8
    assert compact_level(pattern(ci.reshape(-1)), tiny, 2.0 ** -22) is None
    assert compact_level(pattern(ci.reshape(-1)), tiny) is not None
    assert compact_level(pattern(ci.reshape(-1)), torch.zeros_like(v)) is None
    ci[n - 1, 0] -= 1
    assert compact_level(pattern(ci.reshape(-1)), v) is None
