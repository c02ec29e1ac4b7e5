"""coo_to_csr_for_spmv on CPU tensors: torch operations only, no native library."""

import torch

from flagsparse_public_amd import _lib
from flagsparse_public_amd.sparse_operations.spmv_csr import coo_to_csr_for_spmv


def test_no_library_is_loaded(monkeypatch):
    def no_library():
        raise AssertionError("the native library is not for CPU tensors")
    monkeypatch.setattr(_lib, "load", no_library)
    r, c = torch.tensor([2, 0, 2, 1]), torch.tensor([1, 1, 0, 1])
    d, cols, ip = coo_to_csr_for_spmv(torch.tensor([1.0, 2.0, 3.0, 4.0]), r, c, (3, 2))
    assert d.tolist() == [2.0, 4.0, 3.0, 1.0] and cols.tolist() == [1, 1, 0, 1]
    assert ip.tolist() == [0, 1, 2, 4]
