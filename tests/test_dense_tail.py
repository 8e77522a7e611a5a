"""The dense tail of a hierarchy (waterscapes_amd/levels.py) acts like the
levels it replaces: a V-cycle of the cut hierarchy equals the restatement's
V-cycle of the full one (CPU, FP64).  The bound is FP64 round-off grown by
the products that form the tail (a few hundred terms each)."""
import numpy as np
import pytest
import scipy.sparse as sp

from test_batch_pack import _laplacian
from oracle.vcycle import vcycle


@pytest.mark.parametrize("deg,levdeg", [(2, ()), (3, (1,)), (1, ()), (2, (3, 1))])
@pytest.mark.parametrize("rows,masked", [(10**6, True), (10**6, False), (200, True), (1, True)])
def test_cut_hierarchy_equals_full(deg, levdeg, rows, masked):
    from waterscapes_amd import amg, levels as lv
    from waterscapes_amd.amg import AmgParams
    import torch
    prm = AmgParams(max_coarse=12, smoother_degree=deg, level_degrees=levdeg)
    A = _laplacian(9, 0.1)
    n = A.shape[0]
    mask = np.zeros(n, dtype=bool)
    if masked:                       # eliminated rows and columns, as the solver's
        mask[::7] = True
        free = sp.diags((~mask).astype(float))
        A = (free @ A @ free + sp.diags(mask.astype(float))).tocsr()
        A.sort_indices()
    levels, cinv = amg.setup_host(A.indptr, A.indices, A.data, prm)
    assert len(levels) >= 3
    cut, M = lv.with_dense_tail(levels, cinv, rows, prm, "cpu",
                                mask0=torch.as_tensor(mask) if masked else None)
    sizes = [l["n"] for l in levels]
    start = next((i for i, k in enumerate(sizes) if k <= rows), len(sizes) - 1)
    M = lv.host_array(M)
    assert [l["n"] for l in cut] == sizes[:start + 1] and M.shape == (sizes[start],) * 2
    b = np.random.default_rng(0).standard_normal((n, 3))
    b[mask] = 0.0
    A0 = sp.csr_matrix((levels[0]["A_v"], levels[0]["A_ci"], levels[0]["A_rp"]), shape=(n, n))
    ref = vcycle(levels, cinv, A0, mask, prm, b)
    got = vcycle(cut, M, A0, mask, prm, b)
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()


def test_first_level_limit_and_rows():
    from waterscapes_amd import amg, levels as lv
    from waterscapes_amd.amg import AmgParams
    prm = AmgParams(max_coarse=12)
    A = _laplacian(6)
    levels, cinv = amg.setup_host(A.indptr, A.indices, A.data, prm)
    cut, M = lv.with_dense_tail(levels, cinv, 10**6, prm, "cpu", first=1)
    assert len(cut) == 2 and M.shape[0] == levels[1]["n"]
    one, same = lv.with_dense_tail(levels[-1:], cinv, 10**6, prm, "cpu", first=1)
    assert one == levels[-1:] and same is cinv
    assert lv.dense_rows(4, 64 << 20) == 4096 and lv.dense_rows(8, 64 << 20) == 2896


def test_column_ranges():
    """The two column runs the dense pressure kernels read of each row: all
    nonzeros, without the longest run of zeros between two of them."""
    import torch
    from waterscapes_amd import levels as lv
    rng = np.random.default_rng(3)
    M = np.zeros((12, 12))
    M[:4, :4] = rng.standard_normal((4, 4))
    M[4:, 4:] = rng.standard_normal((8, 8))
    M[2] = 0.0
    M[0, 10] = 1.0                       # a second run
    M[6, 4] = M[7, 11] = M[8, 6] = 0.0   # shorter, and an inner zero
    got = lv.column_ranges(torch.as_tensor(M)).numpy()
    want = np.tile([4, 12, 12, 12], (12, 1))
    want[:4] = (0, 4, 4, 4)
    want[0] = (0, 4, 10, 11)
    want[2] = 0
    want[6, 0] = 5
    want[7, 1:] = 11
    want[8] = (4, 6, 7, 12)
    assert np.array_equal(got, want)
