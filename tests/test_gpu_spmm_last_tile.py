"""SpMM with contiguous rows per XCD over several column tiles, the last of a few
columns: around the widths where that begins and ends, with block counts that eight
does not divide; whole-number inputs, exact results."""

import numpy as np
import pytest
import torch

from flagsparse_public_amd import flagsparse_spmm_csr

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("dtype,n_dense", [
    (torch.float32, 257), (torch.float32, 288), (torch.float32, 289), (torch.float32, 513),
    (torch.float64, 129), (torch.float64, 144), (torch.float64, 145), (torch.float64, 257),
    (torch.bfloat16, 513), (torch.float16, 577), (torch.complex64, 129), (torch.complex64, 136),
    (torch.complex128, 65)], ids=str)
@pytest.mark.parametrize("rows", [1, 7, 33, 259, 1001])
def test_rows(rows, dtype, n_dense):
    n_cols = 900
    rng = np.random.default_rng(rows)
    lens = rng.integers(0, 25, rows)
    lens[::97] = 300  # a long row among them
    ip = np.concatenate([[0], np.cumsum(lens)])
    cols, vals = rng.integers(0, n_cols, ip[-1]), rng.integers(-1, 2, ip[-1])
    B = rng.integers(-1, 2, (n_cols, n_dense))
    A = np.zeros((rows, n_cols))
    np.add.at(A, (np.repeat(np.arange(rows), lens), cols), vals)
    f = lambda a, t: torch.from_numpy(a).to(t).to(DEV)  # noqa: E731
    got = flagsparse_spmm_csr(f(vals, dtype), f(cols, torch.int32), f(ip, torch.int64), f(B, dtype),
                              (rows, n_cols))
    want = A @ B  # |sums| < 256: exact in every type
    assert np.array_equal((got.real if dtype.is_complex else got).double().cpu().numpy(), want)
    assert not dtype.is_complex or bool((got.imag == 0).all())
