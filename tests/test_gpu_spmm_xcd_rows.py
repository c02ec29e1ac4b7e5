"""SpMM with contiguous rows per XCD: around the sizes where that begins, with
block counts that eight does not divide; whole-number inputs, exact results."""

import numpy as np
import pytest
import torch

from flagsparse_public_amd import flagsparse_spmm_csr

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("dtype,n_dense", [(torch.float32, 100), (torch.float64, 40)], ids=str)
@pytest.mark.parametrize("rows", [1, 5, 32, 33, 255, 257, 3001])
@pytest.mark.parametrize("past", [0, 1])
def test_rows(rows, dtype, n_dense, past):
    n_cols = (24 << 20) // (n_dense * dtype.itemsize) + past
    rng = np.random.default_rng(rows)
    ip = np.arange(rows + 1) * 12
    cols, vals = rng.integers(0, n_cols, ip[-1]), rng.integers(-2, 3, ip[-1])
    B = torch.randint(-2, 3, (n_cols, n_dense), device=DEV).to(dtype)
    f = lambda a, t: torch.from_numpy(a).to(t).to(DEV)  # noqa: E731
    c = f(cols, torch.int32)
    got = flagsparse_spmm_csr(f(vals, dtype), c, f(ip, torch.int32), B, (rows, n_cols))
    want = (f(vals, dtype)[:, None] * B[c.long()]).view(rows, 12, n_dense).sum(1)
    assert torch.equal(got, want)
