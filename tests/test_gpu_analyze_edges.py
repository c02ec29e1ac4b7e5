"""fs_csr_analyze at the edges of its loads: 64-bit columns at both halves of a
16-byte line with the extreme column at the head, the body and the tail, row
counts around a wavefront, and columns that are all negative.  Exact."""

import numpy as np
import pytest
import torch

from tests.test_gpu_analyze import _expected as _counts
from tests.test_gpu_analyze import _run

pytestmark = pytest.mark.gpu


def _expected(ip, cols):
    st = _counts(ip, cols)
    st[4] = max(st[4], -1)  # the maximum starts at -1, so negative columns leave it there
    return st


@pytest.mark.parametrize("nnz", [0, 1, 2, 3, 4, 31, 2048, 70_001])
@pytest.mark.parametrize("offset", [0, 1])
def test_wide_columns(nnz, offset):
    rng = np.random.default_rng(nnz + offset)
    ip = np.array([0, nnz // 3, nnz], np.int64)
    for place in {0, nnz // 2, nnz - 1}:
        cols = rng.integers(5, 1000, nnz).astype(np.int64)
        if nnz:
            cols[place] = -3
        assert _run(ip, cols, offset, 1000, torch.int64, torch.int64) == _expected(ip, cols).tolist()
        if nnz:
            cols[place] = 1 << 45
        assert _run(ip, cols, offset, 1000, torch.int64, torch.int32) == _expected(ip, cols).tolist()


@pytest.mark.parametrize("n", [1, 63, 64, 65, 4096, 4097, 300_001])
@pytest.mark.parametrize("ptr_dtype", [torch.int32, torch.int64])
def test_row_counts(n, ptr_dtype):
    rng = np.random.default_rng(n)
    lens = rng.integers(0, 6, n)
    lens[rng.integers(0, n)] = 0
    lens[n - 1] = 5000  # the longest row last
    ip = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    cols = np.full(ip[-1], 2, np.int32)
    assert _run(ip, cols, 0, 9, torch.int32, ptr_dtype) == _expected(ip, cols).tolist()


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_only_negative_columns(dtype):
    ip = np.array([0, 40, 100], np.int64)
    cols = np.arange(-100, 0).astype(np.int64 if dtype == torch.int64 else np.int32)
    got = _run(ip, cols, 0, 10, dtype, torch.int32)
    assert got[3] == -100 and got[4] == -1
