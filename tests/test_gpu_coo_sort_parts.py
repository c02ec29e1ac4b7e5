"""fs_coo_sort above 2^22 entries, where the entries are first moved into parts:
the size at which that begins, skewed rows, rows and pairs that span parts, all
value sizes, and the range flags.  Exact, against numpy."""

import numpy as np
import pytest
import torch

from flagsparse_public_amd import _lib
from tests.test_gpu_coo_sort import DEV, _check, _entries

pytestmark = pytest.mark.gpu
FIRST = (1 << 22) + 1  # three parts


@pytest.mark.parametrize("kind,nnz,n,m", [
    ("uniform", FIRST, 300_001, 1 << 20), ("skewed", FIRST, 501, 1201),
    ("repeats", FIRST, 1000, 7), ("sorted", 6_000_000, 3, 1 << 20),
])
def test_order_and_row_pointer(kind, nnz, n, m):
    _check(*_entries(kind, nnz, n, m, 1), n, m)


@pytest.mark.parametrize("idx,dtype", [(torch.int64, torch.int16), (torch.int64, torch.float64),
                                       (torch.int32, torch.complex128)])
def test_types(idx, dtype):
    r, c = _entries("uniform", FIRST, 70_000, 900, 2)
    _check(r, c, 70_000, 900, idx, dtype, out_idx=torch.int32, want_rows=idx == torch.int64,
           ptr=torch.int32)


def test_flags():
    r, c = _entries("uniform", FIRST, 1000, 1000, 3)
    for at, rr, cc, want in ((0, -1, 5, 1), (FIRST - 1, 5, 1000, 2), (FIRST // 2, 1000, -1, 3)):
        r2, c2 = r.copy(), c.copy()
        r2[at], c2[at] = rr, cc
        f = torch.zeros(1, dtype=torch.int64, device=DEV)
        _lib.coo_sort(torch.zeros(FIRST, device=DEV), torch.from_numpy(r2).to(torch.int32).to(DEV),
                      torch.from_numpy(c2).to(torch.int32).to(DEV), 1000, 1000, f)
        assert int(f) & 3 == want
