"""The SpMM row-split rule: the short bound follows twice the mean row length
between its limits, and underfilled launches of long rows go to wavefronts."""

import pytest

from flagsparse_public_amd.rowsplit import SPMM_FILL_LANES, default_spmm_schedule


@pytest.mark.parametrize("mean, short", [(0, 32), (3, 32), (16, 32), (16.5, 64), (32, 64),
                                         (33, 128), (60, 128), (100, 256), (300, 1024),
                                         (513, 1024), (5000, 1024)])
def test_short_bound_follows_the_mean(mean, short):
    n = 1_000_000
    s = default_spmm_schedule(n, int(n * mean), 64)
    assert (s.short_max, s.chunk_nnz) == (short, 256)


@pytest.mark.parametrize("n_dense, lanes", [(1, 8), (8, 8), (32, 8), (33, 16), (64, 16), (128, 32),
                                            (256, 64), (4096, 64)])
def test_underfilled_long_rows_get_wavefronts(n_dense, lanes):
    edge = SPMM_FILL_LANES // lanes
    assert default_spmm_schedule(edge - 1, (edge - 1) * 64, n_dense).short_max == 32
    assert default_spmm_schedule(edge - 1, (edge - 1) * 64, n_dense).chunk_nnz == 512
    assert default_spmm_schedule(edge, edge * 64, n_dense).short_max == 128
    # short rows stay with the lane groups however few they are
    assert default_spmm_schedule(100, 6300, n_dense).chunk_nnz == 256


def test_empty_matrix():
    assert default_spmm_schedule(0, 0, 8).chunk_nnz % 64 == 0
