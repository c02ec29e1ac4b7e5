"""The CSR form of a prepared COO matrix where two threads make their first
products with it at once."""

import torch

from flagsparse_public_amd.sparse_operations import spmv_coo, spmv_csr


def test_another_thread_takes_the_sorted_order_first(monkeypatch):
    d, r, c = torch.ones(2), torch.tensor([0, 1]), torch.tensor([0, 0])

    class Prepared(spmv_coo.PreparedCoo):
        """Its sorted order is there when it is first looked at, and gone after."""
        __slots__ = ("looks",)

        @property
        def _ordered(self):
            self.looks += 1
            return None if self.looks > 1 else spmv_coo._sorted_order(
                (d, r, c), torch.tensor([0, 1, 2]), None, [0] * 16, None)

        @_ordered.setter
        def _ordered(self, value):
            self.looks = 0

    p = Prepared(d, r, c, (2, 1))
    monkeypatch.setattr(spmv_csr, "prepare_spmv_csr", lambda *a, **k: ("csr", a[2].tolist()))
    assert spmv_coo._csr_of(p) == ("csr", [0, 1, 2])
    assert p._csr == ("csr", [0, 1, 2])
