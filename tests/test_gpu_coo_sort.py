"""fs_coo_sort against numpy's stable lexicographic order: sizes around the
tiles, buckets and groups, skewed rows, repeated pairs (equal pairs keep their input
order), index and value types, and the range flags.  Exact."""

import numpy as np
import pytest
import torch

from flagsparse_public_amd import _lib

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _entries(kind, nnz, n, m, seed):
    rng = np.random.default_rng(seed)
    if kind == "uniform":
        r, c = rng.integers(0, n, nnz), rng.integers(0, m, nnz)
    elif kind == "skewed":  # half the entries in two rows, the rest spread
        r = np.where(rng.random(nnz) < 0.5, rng.integers(0, 2, nnz) * (n - 1), rng.integers(0, n, nnz))
        c = rng.integers(0, m, nnz)
    elif kind == "sorted":
        r, c = np.sort(rng.integers(0, n, nnz)), rng.integers(0, m, nnz)
    else:  # "repeats": few distinct pairs, up to hundreds of copies each
        k = max(1, nnz // 200)
        r, c = rng.integers(0, n, k)[rng.integers(0, k, nnz)], np.zeros(nnz, np.int64)
    return r.astype(np.int64), c.astype(np.int64)


def _check(r, c, n, m, idx=torch.int32, dtype=torch.int32, out_idx=None, want_rows=True,
           ptr=torch.int64):
    nnz = r.size
    # the values are the input positions, so they show the order itself
    vals = torch.arange(nnz, dtype=torch.int64).to(dtype)
    flags = torch.full((1,), 99, dtype=torch.int64, device=DEV)
    d, kr, kc, ip = _lib.coo_sort(vals.to(DEV), torch.from_numpy(r).to(idx).to(DEV),
                                  torch.from_numpy(c).to(idx).to(DEV), n, m, flags,
                                  index_dtype=out_idx, want_rows=want_rows, ptr_dtype=ptr)
    assert flags.item() == 0
    order = np.lexsort((np.arange(nnz), c, r))
    assert torch.equal(d.cpu(), vals[torch.from_numpy(order)])
    assert kc.dtype == (out_idx or idx) and np.array_equal(kc.cpu().numpy(), c[order])
    if want_rows:
        assert np.array_equal(kr.cpu().numpy(), r[order])
    want = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))])
    assert ip.dtype == ptr and np.array_equal(ip.cpu().numpy(), want)


@pytest.mark.parametrize("nnz", [1, 2, 7, 8, 9, 1023, 1024, 1025, 2049, 8191, 8193, 100_003])
@pytest.mark.parametrize("kind", ["uniform", "skewed", "sorted", "repeats"])
def test_order_and_row_pointer(nnz, kind):
    n, m = 501, 1201
    _check(*_entries(kind, nnz, n, m, nnz), n, m)


@pytest.mark.parametrize("kind", ["uniform", "skewed", "repeats"])
def test_largest_size(kind):
    """The size limit, where groups are largest, with all 64 key bits in use."""
    n, m = 1 << 20, 1 << 22
    _check(*_entries(kind, 1 << 22, n, m, 3), n, m)


def test_sizes_that_do_not_apply():
    ok = _lib.coo_sort_applies
    assert ok(7 << 24, 5, 5) and not ok((7 << 24) + 1, 5, 5) and not ok(0, 5, 5)
    assert ok(1 << 22, 1 << 21, 1 << 21) and not ok(1 << 22, 1 << 21, (1 << 21) + 1)
    assert ok(5, 2**31 - 1, 1 << 30) and not ok(5, 2**31, 5) and not ok(5, 5, 2**31)


@pytest.mark.parametrize("idx", [torch.int32, torch.int64])
@pytest.mark.parametrize("out_idx", [torch.int32, torch.int64])
@pytest.mark.parametrize("dtype", [torch.int16, torch.int32, torch.float64, torch.complex128])
def test_types(idx, out_idx, dtype):
    r, c = _entries("uniform", 20_000, 3000, 70, 5)
    _check(r, c, 3000, 70, idx, dtype, out_idx, want_rows=out_idx == torch.int64, ptr=torch.int32)


def test_empty_rows_at_both_ends():
    r = np.array([5, 5, 9, 5], np.int64)
    _check(r, np.array([3, 1, 0, 3], np.int64), 20_000, 4)


@pytest.mark.parametrize("idx", [torch.int32, torch.int64])
def test_flags(idx):
    r, c = _entries("uniform", 30_000, 100, 50, 6)
    v = torch.zeros(r.size, device=DEV)

    def flag(rr, cc, n=100, m=50):
        f = torch.zeros(1, dtype=torch.int64, device=DEV)
        _lib.coo_sort(v, torch.from_numpy(rr).to(idx).to(DEV), torch.from_numpy(cc).to(idx).to(DEV),
                      n, m, f)
        return f.item()

    def put(a, value):
        a = a.copy()
        a[12_345] = value
        return a
    assert flag(r, c) == 0
    for bad in (-1, 100) + ((1 << 40, -(1 << 40)) if idx == torch.int64 else ()):
        assert flag(put(r, bad), c) == _lib.COO_BAD_ROW
    for bad in (-7, 50):
        assert flag(r, put(c, bad)) == _lib.COO_BAD_COL
    assert flag(put(r, 100), put(c, 50)) == _lib.COO_BAD_ROW | _lib.COO_BAD_COL


def test_operators_beyond_the_sort():
    """Sizes past the key's 64 bits take the general path: same results."""
    from flagsparse_public_amd import flagsparse_spmm_coo, flagsparse_spmv_coo
    from flagsparse_public_amd.sparse_operations.spmv_csr import coo_to_csr_for_spmv
    rng = np.random.default_rng(0)
    n, m, nnz = 50, (1 << 30) + 1, 1 << 20
    assert not _lib.coo_sort_applies(nnz, 1 << 14, m)
    r, c = rng.integers(0, 1 << 14, nnz), rng.integers(0, n, nnz)
    d, cols, ip = coo_to_csr_for_spmv(torch.arange(nnz, device=DEV), torch.from_numpy(r).to(DEV),
                                      torch.from_numpy(c).to(DEV), (1 << 14, m))
    order = np.lexsort((np.arange(nnz), c, r))
    assert np.array_equal(d.cpu().numpy(), order) and np.array_equal(cols.cpu().numpy(), c[order])
    # one entry more than the limit, few columns: whole numbers, so exact
    nnz = (1 << 22) + 1
    r, c = rng.integers(0, n, nnz), rng.integers(0, n, nnz)
    v = rng.integers(-4, 5, nnz).astype(np.float64)
    x = np.arange(n, dtype=np.float64)
    A = np.zeros((n, n))
    np.add.at(A, (r, c), v)
    args = [torch.from_numpy(a).to(DEV) for a in (v, r, c)]
    assert np.array_equal(flagsparse_spmv_coo(*args, torch.from_numpy(x).to(DEV), (n, n)).cpu(), A @ x)
    C = flagsparse_spmm_coo(*args, torch.from_numpy(np.stack([x, -x], 1)).to(DEV), (n, n))
    assert np.array_equal(C.cpu().numpy(), np.stack([A @ x, -(A @ x)], 1))


@pytest.mark.parametrize("sort_by_row", [True, False])
def test_prepared_fields(sort_by_row):
    from flagsparse_public_amd import prepare_spmv_coo
    r, c = _entries("skewed", 5000, 300, 200, 8)
    v = torch.rand(r.size, device=DEV)
    p = prepare_spmv_coo(v, torch.from_numpy(r).to(DEV), torch.from_numpy(c).to(torch.int32).to(DEV),
                         (300, 200), sort_by_row=sort_by_row)
    order = torch.from_numpy(np.lexsort((np.arange(r.size), c, r)))
    assert p.row.dtype == p.col.dtype == torch.int64
    assert np.array_equal(p.row.cpu(), r[order]) and np.array_equal(p.col.cpu(), c[order])
    assert torch.equal(p.data.cpu(), v.cpu()[order])
    if not sort_by_row:
        assert p.seg_starts is None and p.n_segs == 0 and not p.use_seg_kernel
        return
    rs = np.sort(r)
    starts = np.concatenate([[0], np.nonzero(rs[1:] != rs[:-1])[0] + 1, [r.size]])
    assert p.use_seg_kernel and p.n_segs == starts.size - 1
    assert np.array_equal(p.seg_starts.cpu().numpy(), starts)
