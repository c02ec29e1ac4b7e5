"""Sizes that fs_csr_analyze_split refuses before it launches anything: its packed
count holds fewer than 2^27 long rows."""

import ctypes

import pytest

from flagsparse_public_amd import _lib

BIG = 1 << 27


def _call(n_rows, cap_long, nnz=2**31 - 1):
    """On addresses that nothing may be read from or written to."""
    lib = _lib.load()
    csr = _lib.FsCsr(value_type=_lib.FS_F32, index_type=_lib.FS_I32, ptr_type=_lib.FS_I32,
                     reserved=0, n_rows=n_rows, n_cols=5, nnz=nnz, row_ptr=64, col_idx=64,
                     values=None)
    rc = lib.fs_csr_analyze_split(ctypes.byref(csr), 64, 1, 64, 64, 64, cap_long, 64, 100, None, None)
    return rc, lib.fs_last_error().decode()


@pytest.mark.parametrize("n_rows,cap_long", [(BIG, BIG), (2**30, 2**30), (2**31 - 1, BIG),
                                             (BIG, 2**31 - 1)])
def test_too_many_long_rows(n_rows, cap_long):
    rc, msg = _call(n_rows, cap_long)
    assert rc == _lib.FS_ERR_UNSUPPORTED and "2^27" in msg


def test_plans_list_such_rows_otherwise():
    fits = _lib.splits_natively
    assert not fits(2**31 - 1, 2**31 - 1, 1) and not fits(2 * BIG, BIG, 1)
    assert fits(2 * BIG - 1, 2**31 - 1, 1) and fits(2**31 - 1, BIG - 1, 1)
    assert fits(2**31 - 1, 2**31 - 1, 32) and not fits(2**31, 10, 32)
