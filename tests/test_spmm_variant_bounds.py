"""The row split of a library-chosen SpMM variant: rows that the variant itself cuts
into chunks, whose sums are compensated in fp32, stay in chunks."""

import types

import pytest
import torch

from flagsparse_public_amd.autotune import SPMM_VARIANTS
from flagsparse_public_amd.sparse_operations.spmm_csr import spmm_launch_schedule


@pytest.mark.parametrize("mean", [10, 40, 100, 300])
@pytest.mark.parametrize("n_dense", [8, 64, 256])
@pytest.mark.parametrize("variant", SPMM_VARIANTS, ids=lambda v: f"{v.short_max}_{v.col_tile}_{v.xcd_remap}")
def test_chosen_variants_keep_their_chunked_rows(variant, mean, n_dense):
    n_rows = 100_000
    data = types.SimpleNamespace(numel=lambda: n_rows * mean, element_size=lambda: 4,
                                 dtype=torch.float32)
    p = types.SimpleNamespace(schedule=variant, library_schedule=True, n_rows=n_rows, data=data,
                              max_row_nnz=4 * mean, _plans={})
    sch, _ = spmm_launch_schedule(p, n_dense)
    assert sch.short_max <= min(256, variant.short_max)
