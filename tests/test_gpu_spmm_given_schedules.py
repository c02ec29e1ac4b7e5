"""Which SpMM launches leave the block order and the column tiles to the launch's
own rules: those of schedules that the library chose.  A caller's run as given."""

import pytest
import torch

from flagsparse_public_amd import (flagsparse_spmm_csr, flagsparse_spmm_csr_opt,
                                   flagsparse_spmm_csr_opt_alg2, prepare_spmm_csr_opt,
                                   prepare_spmm_csr_opt_alg2)
from flagsparse_public_amd import _lib
from flagsparse_public_amd.rowsplit import Schedule

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.fixture
def launched(monkeypatch):
    """xcd_remap of every SpMM plan that is launched."""
    seen = []
    spmm = _lib.spmm

    def record(csr, B, ldb, C, ldc, n, alpha, beta, plan, col_tile, device):
        seen.append((plan.xcd_remap, col_tile))
        return spmm(csr, B, ldb, C, ldc, n, alpha, beta, plan, col_tile, device)
    monkeypatch.setattr(_lib, "spmm", record)
    return seen


def _args():
    ptr = torch.arange(101, device=DEV) * 4
    cols = torch.arange(400, device=DEV, dtype=torch.int32) % 50
    return torch.ones(400, device=DEV), cols, ptr, torch.ones((50, 64), device=DEV), (100, 50)


@pytest.mark.parametrize("xcd", [0, 1])
def test_given(launched, xcd):
    data, cols, ptr, B, shape = _args()
    sch = Schedule(group_lanes=1, short_max=64, chunk_nnz=128, xcd_remap=xcd)
    p = prepare_spmm_csr_opt(data, cols, ptr, shape, schedule=sch)
    flagsparse_spmm_csr_opt(B=B, prepared=p)
    flagsparse_spmm_csr_opt_alg2(B=B, prepared=prepare_spmm_csr_opt_alg2(data, cols, ptr, shape,
                                                                        schedule=sch))
    assert launched == [(xcd, 0)] * 2


def test_library(launched):
    data, cols, ptr, B, shape = _args()
    flagsparse_spmm_csr(data, cols, ptr, B, shape)
    flagsparse_spmm_csr_opt(B=B, prepared=prepare_spmm_csr_opt(data, cols, ptr, shape,
                                                              schedule="default"))
    flagsparse_spmm_csr_opt_alg2(B=B, prepared=prepare_spmm_csr_opt_alg2(data, cols, ptr, shape,
                                                                        schedule="default"))
    assert [x for x, _ in launched] == [_lib.FS_XCD_AUTO] * 3
