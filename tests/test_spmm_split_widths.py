"""spmm_splits lists every split that the rule gives a matrix, and few others."""

import pytest

from flagsparse_public_amd.rowsplit import default_spmm_schedule, spmm_splits


@pytest.mark.parametrize("item", [2, 4, 8, 16])
@pytest.mark.parametrize("longest", [1, 3, 100])  # in mean row lengths
@pytest.mark.parametrize("n_rows,nnz", [(1, 0), (10, 40), (300, 60_000), (900, 270_000),
                                        (900, 360_000), (3000, 30_000), (5000, 500_000),
                                        (15_000, 1_048_575), (30_000, 1_048_575),
                                        (30_000, 6_000_000), (40_000, 4_000_000),
                                        (200_000, 1_000_000), (1_000_000, 15_000_000)])
def test_all_splits_are_listed(item, longest, n_rows, nnz):
    step = list(range(1, 3000)) + [2**k + d for k in range(12, 28) for d in (-1, 0, 1)]
    max_row = longest * nnz // n_rows
    of = [default_spmm_schedule(n_rows, nnz, n, item, max_row=max_row) for n in step]
    splits = spmm_splits(n_rows, nnz, item)
    assert {(s.short_max, s.chunk_nnz) for s in of} <= set(splits)
    assert len(splits) == len(set(splits)) <= 5
    if nnz >= 1 << 20 and (n_rows >= 1 << 18 or nnz < 64 * n_rows):
        assert len(splits) == 1  # large matrices plan once
