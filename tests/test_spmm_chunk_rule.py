"""The chunk size of default_spmm_schedule: smaller where B rows are wide and the
launch gathers little, unchanged elsewhere."""

import pytest

from flagsparse_public_amd.rowsplit import SPMM_CHUNK_BYTES, default_spmm_schedule


@pytest.mark.parametrize("n_dense, item, nnz, chunk", [
    (32, 4, 1000, 256),                                 # 128-byte B rows: eight lanes
    (33, 4, 1000, 128), (64, 4, 1000, 128),
    (65, 4, 1000, 64), (160, 2, 1000, 64), (24, 8, 1000, 128), (128, 16, 1000, 64),
    (128, 4, SPMM_CHUNK_BYTES // 1024 - 1, 64), (128, 4, SPMM_CHUNK_BYTES // 1024, 128),
    (128, 4, SPMM_CHUNK_BYTES // 512 - 1, 128), (128, 4, SPMM_CHUNK_BYTES // 512, 256),
    (128, 0, 1000, 256),                                # item size not given
])
def test_chunk_follows_the_gathered_bytes(n_dense, item, nnz, chunk):
    s = default_spmm_schedule(10_000_000, nnz, n_dense, item)
    assert (s.chunk_nnz, s.short_max) == (chunk, 32)
