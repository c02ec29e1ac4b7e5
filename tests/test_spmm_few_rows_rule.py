"""The SpMM row split where every row may get a wavefront: rows of like length only
as long as the lanes added are few against the entries, skewed rows as before, and
chunk sizes there."""

import types

import pytest
import torch

from flagsparse_public_amd.autotune import SPMM_VARIANTS
from flagsparse_public_amd.rowsplit import (SPMM_EVEN_ROWS, default_spmm_schedule, spmm_row_lanes,
                                            spmm_splits)
from flagsparse_public_amd.sparse_operations.spmm_csr import spmm_launch_schedule


def _split(n_rows, mean, n_dense, item, longest, wide=False):
    s = default_spmm_schedule(n_rows, n_rows * mean, n_dense, item, wide, longest)
    return s.short_max, s.chunk_nnz


@pytest.mark.parametrize("n_rows,mean,n_dense,item,few", [
    (30_000, 200, 8, 4, True), (30_000, 100, 8, 4, False), (15_000, 100, 8, 4, True),
    (15_000, 70, 8, 4, False), (5000, 70, 64, 4, True), (15_000, 100, 64, 4, False),
    (15_000, 100, 8, 8, False), (15_000, 200, 8, 8, True), (30_000, 100, 1, 8, True),
    (8000, 200, 36, 8, False), (1500, 100, 256, 4, False), (300, 200, 256, 4, True),
    (5000, 63, 8, 4, False), (100_000, 200, 8, 4, False)])
def test_rows_of_like_length(n_rows, mean, n_dense, item, few):
    longest = SPMM_EVEN_ROWS * mean
    assert (_split(n_rows, mean, n_dense, item, longest)[0] == 32) == few
    # skewed rows and unknown ones get wavefronts wherever the groups leave the chip unfilled
    wider = mean >= 64 and n_rows * max(8, n_dense // 4) < 1 << 18
    for row in (longest + 1, None):
        assert (_split(n_rows, mean, n_dense, item, row)[0] == 32) == wider


@pytest.mark.parametrize("item", [2, 4, 8, 16])
@pytest.mark.parametrize("n_dense", [1, 4, 8, 64, 65, 256])
@pytest.mark.parametrize("mean", [100, 320, 321, 1000])
def test_chunks_there(item, n_dense, mean):
    narrow = n_dense * item <= 16
    long = item <= 4 and n_dense * item <= 256 and (mean <= 320 or narrow)
    assert _split(300, mean, n_dense, item, None) == (32, 512 if long else 256)


@pytest.mark.parametrize("n_rows,most", [(300, 256), (5000, 1024)])
def test_wide_sums_keep_long_chains_where_the_chip_is_filled(n_rows, most):
    """fp32 values summed in fp64: rows of 400 to 600."""
    assert _split(n_rows, 512, 300, 4, None, wide=True)[0] == (most if most == 1024 else 32)
    assert _split(100_000, 512, 300, 4, None, wide=True)[0] == 1024
    assert _split(100_000, 512, 300, 4, None)[0] == 256


@pytest.mark.parametrize("n_dense,item,lanes", [(1, 4, 1), (3, 4, 4), (8, 4, 8), (9, 4, 16),
                                                (16, 4, 8), (32, 4, 8), (33, 4, 16), (130, 4, 64),
                                                (300, 4, 128), (8, 8, 8), (36, 8, 32), (130, 8, 128),
                                                (64, 2, 8), (256, 2, 32), (5, 16, 8)])
def test_lanes_of_a_row(n_dense, item, lanes):
    assert spmm_row_lanes(n_dense, item) == lanes


def _launch(variant, n_rows, mean, n_dense, dtype=torch.float32):
    data = types.SimpleNamespace(numel=lambda: n_rows * mean, element_size=lambda: dtype.itemsize,
                                 dtype=dtype)
    p = types.SimpleNamespace(schedule=variant, library_schedule=True, n_rows=n_rows, data=data,
                              max_row_nnz=2 * mean, _plans={})
    return spmm_launch_schedule(p, n_dense)


def test_a_lowered_bound_keeps_the_variants_chunks():
    """Rows over 64 entries in chunks of 64 would all need two and a fix-up."""
    lower = next(v for v in SPMM_VARIANTS if v.short_max == 64)
    sch, _ = _launch(lower, 300, 60, 130)
    assert (sch.short_max, sch.chunk_nnz) == (64, lower.chunk_nnz) and lower.chunk_nnz >= 128
    assert _split(300, 60, 130, 4, 120) == (128, 64)
    assert (128, 64) in spmm_splits(300, 300 * 60, 4)
