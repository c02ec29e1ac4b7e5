"""COO operators where the native sort does not order the entries: keys of more
than 64 bits, and entries that its sample does not suit (flag 4).  Exact."""

import numpy as np
import pytest
import torch

from flagsparse_public_amd import (_lib, flagsparse_spmm_coo, flagsparse_spmv_coo,
                                   prepare_spmv_coo)
from flagsparse_public_amd.sparse_operations.spmv_csr import coo_to_csr_for_spmv

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _dev(*arrays):
    return [torch.from_numpy(np.ascontiguousarray(a)).to(DEV) for a in arrays]


def _check_operators(r, c, n, m, seed):
    """Whole numbers: every order of the sums gives the same result."""
    rng = np.random.default_rng(seed)
    v = rng.integers(-4, 5, r.size).astype(np.float64)
    x = rng.integers(-4, 5, m).astype(np.float64)
    want = np.bincount(r, weights=v * x[c], minlength=n)
    dv, dr, dc, dx = _dev(v, r, c, x)
    assert np.array_equal(flagsparse_spmv_coo(dv, dr, dc, dx, (n, m)).cpu().numpy(), want)
    C = flagsparse_spmm_coo(dv, dr, dc, torch.stack([dx, -dx], 1), (n, m)).cpu().numpy()
    assert np.array_equal(C, np.stack([want, -want], 1))
    order = np.lexsort((np.arange(r.size), c, r))
    p = prepare_spmv_coo(torch.arange(r.size, device=DEV, dtype=torch.float64), dr, dc, (n, m))
    assert np.array_equal(p.data.cpu().numpy(), order)
    rs = np.sort(r)
    starts = np.concatenate([[0], np.nonzero(rs[1:] != rs[:-1])[0] + 1, [r.size]])
    assert p.n_segs == starts.size - 1 and np.array_equal(p.seg_starts.cpu().numpy(), starts)
    d, cols, ip = coo_to_csr_for_spmv(torch.arange(r.size, device=DEV), dr, dc, (n, m))
    assert np.array_equal(d.cpu().numpy(), order) and np.array_equal(cols.cpu().numpy(), c[order])
    assert np.array_equal(ip.cpu().numpy(), np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]))


def test_keys_of_65_bits():
    n, m, nnz = (1 << 22) + 1, 1 << 22, (1 << 19) + 1
    assert not _lib.coo_sort_applies(nnz, n, m) and _lib.coo_sort_applies(nnz, n - 1, m)
    rng = np.random.default_rng(0)
    _check_operators(rng.integers(0, n, nnz), rng.integers(0, m, nnz), n, m, 1)
    r, c = _dev(np.array([0, n]).repeat(nnz // 2), np.zeros(nnz // 2 * 2, np.int64))
    v = torch.ones(r.numel(), device=DEV)
    for bad_r, bad_c in ((r, c), (c, r)):
        shape = (n, m) if bad_r is r else (m, n)
        with pytest.raises(IndexError, match="row" if bad_r is r else "col"):
            flagsparse_spmv_coo(v, bad_r, bad_c, torch.ones(shape[1], device=DEV), shape)
        with pytest.raises(IndexError, match="row" if bad_r is r else "col"):
            flagsparse_spmm_coo(v, bad_r, bad_c, torch.ones((shape[1], 1), device=DEV), shape)


def _sampled(nnz):
    """The places of the sort's sample (one part of several buckets)."""
    n_samples = -(-nnz // 448) * 4
    i = np.arange(n_samples, dtype=np.uint64)
    a, z = i * np.uint64(nnz) // np.uint64(n_samples), (i + 1) * np.uint64(nnz) // np.uint64(n_samples)
    m32 = np.uint64(0xFFFFFFFF)
    h = i * np.uint64(2654435761) & m32
    h = (h ^ (h >> np.uint64(15))) * np.uint64(2246822519) & m32
    return (a + (h ^ (h >> np.uint64(13))) % (z - a)).astype(np.int64)


@pytest.mark.parametrize("nnz", [10_000, 50_001])
def test_a_sample_that_misses_the_rest(nnz):
    """Every sampled entry lies in row 0 and all others behind the last splitter:
    one bucket holds nearly all entries, more than the largest group takes."""
    n, m = 300, 200
    rng = np.random.default_rng(nnz)
    r, c = rng.integers(1, n, nnz), rng.integers(0, m, nnz)
    r[_sampled(nnz)] = 0
    flags = torch.zeros(1, dtype=torch.int64, device=DEV)
    _lib.coo_sort(torch.zeros(nnz, device=DEV), *_dev(r, c), n, m, flags)
    assert flags.item() == _lib.COO_OVERFLOW
    _check_operators(r, c, n, m, 2)
