"""fs_coo_sort where its groups' bins crowd: a long row among short ones (cut a
second time), columns clustered at every scale (merge sort), a sample that falls
into one table slot, and tile edges.  Exact, against numpy."""

import numpy as np
import pytest
import torch

from tests.test_gpu_coo_sort import _check

pytestmark = pytest.mark.gpu


def _long_row(nnz, rng):  # 40% of the entries in short rows, one row takes the rest
    r = np.where(rng.random(nnz) < 0.4, rng.integers(0, 5000, nnz), 2500)
    return r, rng.integers(0, 1 << 20, nnz)


def _clustered(nnz, rng):  # columns log-uniform: half of them below 1024 of 2^20
    return rng.integers(0, 2, nnz), np.exp(rng.random(nnz) * np.log(1 << 20)).astype(np.int64)


def _one_slot(nnz, rng):  # rows at the end of a long range, few columns
    return 4999 - (rng.random(nnz) < 0.01), rng.integers(0, 3, nnz)


@pytest.mark.parametrize("make", [_long_row, _clustered, _one_slot])
@pytest.mark.parametrize("nnz", [600, 8191, 8192, 8193, 60_000])
@pytest.mark.parametrize("dtype", [torch.int16, torch.int32, torch.float64, torch.complex128])
def test_crowded_bins(make, nnz, dtype):
    r, c = make(nnz, np.random.default_rng(nnz))
    _check(r.astype(np.int64), c.astype(np.int64), 5000, 1 << 20, dtype=dtype)
