"""The batch on the cell-wise operator: the checks of test_gpu_batch.py
(operator and preconditioner against the oracle per instance, every step
against the oracle, isolation, inactive instances) with every batch large
enough to run cell by cell, and the FP32 operator against the FP64 one on
instances whose cells do not fill their blocks."""
import numpy as np
import pytest

import test_gpu_batch as base

pytestmark = pytest.mark.gpu

FP32_RTOL = 2e-6     # per field and instance, as the single-instance operator's FP32 check


@pytest.fixture(autouse=True)
def _cells(monkeypatch):
    from waterscapes_amd import batch
    monkeypatch.setattr(batch, "BATCH_CELLS", 1)


def test_operator_and_preconditioner_blocks():
    base.test_batch_operator_and_preconditioner_blocks()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_matches_oracle(precision):
    base.test_batch_matches_oracle(precision)


def test_isolation():
    base.test_batch_isolation()


def test_inactive_instances_untouched():
    base.test_batch_inactive_instances_untouched()


def test_fp32_operator_and_residual():
    import torch
    batch = base._batch(base._make([0, 1, 2]), "mixed")
    assert batch.cells and sum(e.space.mesh.num_cells() for e in batch.engines) % 256
    g = torch.Generator(device="cpu").manual_seed(3)
    x = torch.randn(batch.n, generator=g, dtype=torch.float64).cuda()
    b = torch.randn(batch.n, generator=g, dtype=torch.float64).cuda()
    for rhs in (None, b):
        y64 = batch.unpack(batch.apply(batch.pack(x), None if rhs is None else batch.pack(rhs)))
        y32 = batch.unpack(batch.apply(batch.pack(x.float()),
                                       None if rhs is None else batch.pack(rhs.float()),
                                       dtype=1))
        for k, e in enumerate(batch.engines):
            a = int(batch.n_off[k])
            for f in range(e.space.F + 1):
                i = torch.as_tensor(a + e.space.field_index(f), device="cuda")
                scale = y64[i].abs().max().item()
                assert (y32[i].double() - y64[i]).abs().max().item() <= FP32_RTOL * scale
    batch.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_no_operator_is_refused(precision, monkeypatch):
    """A handle made without packed values, whose cell-wise operator was
    refused, returns an error from solves and applications (no launch)."""
    import torch
    from waterscapes_amd import _lib, batch as B
    monkeypatch.setattr(B.MPETBatch, "_pack_cells", lambda self: B.BatchCellDesc())
    b = B.MPETBatch.__new__(B.MPETBatch)
    with pytest.raises(_lib.MpetError) as ei:
        b.__init__([it[2] for it in base._make([0, 2])], precision=precision)
    invalid = ei.value.code
    x = torch.ones(b.n, dtype=torch.float64, device="cuda")
    for dtype in (0,) if precision == "fp64" else (0, 1):
        with pytest.raises(_lib.MpetError) as ei:
            b.apply(x if dtype == 0 else x.float(), dtype=dtype)
        assert ei.value.code == invalid
    y, stats = torch.zeros_like(x), (B.SolveStats * b.K)()
    rc = B._bind().mpet_batch_solve(b.handle, _lib.ptr(x), _lib.ptr(y), None, stats,
                                    _lib.stream_ptr())
    assert rc == invalid and not y.any()
    b.close()
