"""SpMM with B rows cut into 128-byte tiles: around the sizes where that begins
and ends, whole-number inputs whose products and sums are exact in every type, so
the result must equal the integers."""

import numpy as np
import pytest
import torch

from flagsparse_public_amd import flagsparse_spmm_csr

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
MB = 1 << 20


def _check(n_rows, n_cols, mean, n_dense, dtype, long_rows=0):
    rng = np.random.default_rng(n_cols + n_dense)
    lens = np.full(n_rows, mean)
    lens[rng.permutation(n_rows)[:long_rows]] = 200
    ip = np.concatenate([[0], np.cumsum(lens)])
    cols = rng.integers(0, n_cols, ip[-1])
    vals = rng.integers(-1, 2, ip[-1])
    B = rng.integers(-1, 2, (n_cols, n_dense)).astype(np.int16)
    want = np.add.reduceat(vals[:, None] * B[cols], ip[:-1])  # |sums| <= 200: exact in bfloat16
    t = [torch.from_numpy(a) for a in (vals, cols.astype(np.int32), ip.astype(np.int32), B)]
    got = flagsparse_spmm_csr(t[0].to(dtype).to(DEV), t[1].to(DEV), t[2].to(DEV),
                              t[3].to(dtype).to(DEV), (n_rows, n_cols))
    got = (got.real if dtype.is_complex else got).double().cpu().numpy()
    assert np.array_equal(got, want)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32, torch.float64,
                                   torch.complex64, torch.complex128], ids=str)
@pytest.mark.parametrize("lines", [2, 4, 8])
@pytest.mark.parametrize("edge", ["below", "above", "last", "past"])
def test_sizes_of_b(dtype, lines, edge):
    first, last = 6 * MB // (128 * lines), (8 if lines == 8 else 12) * MB // 128
    n_cols = {"below": first, "above": first + 1, "last": last, "past": last + 1}[edge]
    _check(515, n_cols, 9, 128 * lines // dtype.itemsize, dtype)


@pytest.mark.parametrize("mean,long_rows,n_dense", [(7, 0, 128), (8, 0, 128), (33, 0, 64),
                                                    (9, 8, 128), (9, 9, 128), (9, 0, 127),
                                                    (9, 0, 129), (9, 0, 96)])
def test_other_conditions(mean, long_rows, n_dense):
    _check(1024, 30_000, mean, n_dense, torch.float32, long_rows)
