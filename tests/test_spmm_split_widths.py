"""spmm_splits lists every split that the rule gives a matrix."""

import pytest

from flagsparse_public_amd.rowsplit import default_spmm_schedule, spmm_splits


@pytest.mark.parametrize("item", [2, 4, 8, 16])
@pytest.mark.parametrize("n_rows,nnz", [(1, 0), (10, 40), (900, 270_000), (3000, 30_000),
                                        (5000, 500_000), (30_000, 1_048_575), (40_000, 4_000_000),
                                        (200_000, 1_000_000), (1_000_000, 15_000_000)])
def test_widths_cover_the_splits(item, n_rows, nnz):
    step = list(range(1, 3000)) + [2**k + d for k in range(12, 28) for d in (-1, 0, 1)]
    of = [default_spmm_schedule(n_rows, nnz, n, item) for n in step]
    assert {(s.short_max, s.chunk_nnz) for s in of} == set(spmm_splits(n_rows, nnz, item))
