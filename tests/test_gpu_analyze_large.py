"""Statistics of column arrays on both sides of the size above which the pass
reads them past the caches."""

import numpy as np
import pytest
import torch

from flagsparse_public_amd import _lib

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("idx", [torch.int32, torch.int64])
@pytest.mark.parametrize("past", [0, 1, 3])
@pytest.mark.parametrize("narrow", [False, True])
def test_extremes_found(idx, past, narrow):
    nnz, n = (80 << 20) // idx.itemsize + past, 1000
    ip = torch.linspace(0, nnz, n + 1, dtype=torch.float64, device=DEV).to(torch.int64)
    ip[-1] = nnz
    cols = torch.full((nnz,), 500, dtype=idx, device=DEV)
    cols[nnz // 3], cols[nnz - 1] = 3, 997
    vals = torch.empty(nnz, dtype=torch.float16, device=DEV)
    csr = _lib.make_csr(vals, cols, ip, n, n)
    if narrow:
        stats, *_, c32, _ = _lib.analyze_split(csr, DEV, 1 << 30, 64, idx == torch.int64)
        assert c32 is None or torch.equal(c32, cols.to(torch.int32))
    else:
        stats = _lib.analyze(csr, DEV)
    lens = np.diff(ip.cpu().numpy())
    assert (stats[0], stats[1], stats[3], stats[4]) == (0, nnz, 3, 997)
    assert (stats[5], stats[6]) == (lens.max(), lens.min())
