"""Column tiles of library-chosen fp32 SpMM variants: widths that four columns do
not divide are one tile where the rows fill the chip."""

import types

import pytest
import torch

from flagsparse_public_amd.autotune import SPMM_VARIANTS
from flagsparse_public_amd.sparse_operations.spmm_csr import spmm_launch_schedule


@pytest.mark.parametrize("variant", SPMM_VARIANTS, ids=lambda v: f"{v.short_max}_{v.col_tile}_{v.xcd_remap}")
@pytest.mark.parametrize("n_rows,n_dense,one", [
    (120_000, 66, True), (120_000, 99, True), (120_000, 129, True), (120_000, 258, True),
    (120_000, 64, False), (120_000, 100, False), (120_000, 256, False), (300, 130, False),
    (4095, 129, False), (4096, 129, True)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_tile(variant, n_rows, n_dense, one, dtype):
    data = types.SimpleNamespace(numel=lambda: n_rows * 40, element_size=lambda: dtype.itemsize,
                                 dtype=dtype)
    p = types.SimpleNamespace(schedule=variant, library_schedule=True, n_rows=n_rows, data=data,
                              max_row_nnz=80, _plans={})
    _, tile = spmm_launch_schedule(p, n_dense)
    whole = variant.col_tile * (n_dense // 64 if n_dense > 64 else 1)
    assert tile == (0 if one and dtype == torch.float32 else whole)
