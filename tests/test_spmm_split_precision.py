"""The SpMM row split with the value size given, as every launch gives it: no sum of
one chain gets longer than the types allow."""

import pytest

from flagsparse_public_amd.rowsplit import default_spmm_schedule


@pytest.mark.parametrize("item", [2, 4, 8, 16])
@pytest.mark.parametrize("mean", [0, 16, 60, 129, 300, 1000, 5000])
@pytest.mark.parametrize("n_dense", [1, 16, 64, 256, 1000])
@pytest.mark.parametrize("n_rows", [100, 5000, 100_000])
def test_rows_over_256_entries_are_chunked(item, mean, n_dense, n_rows):
    s = default_spmm_schedule(n_rows, n_rows * mean, n_dense, item)
    assert s.short_max <= 256
    # chunks of 512 only where their sums are compensated or wider than the values
    assert s.chunk_nnz <= (512 if item <= 4 else 256)
