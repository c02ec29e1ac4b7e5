"""COO operators on values that torch holds as lazy views (the conjugate and the
negative bit): the same results as on the values written out.  Exact."""

import numpy as np
import pytest
import torch

from flagsparse_public_amd import flagsparse_spmm_coo, flagsparse_spmv_coo, prepare_spmv_coo
from flagsparse_public_amd.sparse_operations.spmv_csr import coo_to_csr_for_spmv

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
N = 300


def _entries(nnz):
    rng = np.random.default_rng(nnz)
    r, c = rng.integers(0, N, nnz), rng.integers(0, N, nnz)
    if nnz == 1:  # one entry: a strided view of it counts as contiguous
        r[:], c[:] = 7, 3
    z = rng.integers(-4, 5, nnz) + 1j * rng.integers(1, 5, nnz)  # whole numbers: sums are exact
    return (torch.from_numpy(z).to(DEV), torch.from_numpy(r).to(DEV), torch.from_numpy(c).to(DEV))


def _view(kind, nnz, dtype):
    z, r, c = _entries(nnz)
    if kind == "conj":
        v = z.to(dtype).conj()
        assert v.is_conj()
    else:
        v = torch._neg_view(z.imag.contiguous().to(dtype)) if nnz > 1 else z.to(
            torch.complex64 if dtype == torch.float32 else torch.complex128).conj().imag
        assert v.is_neg() and v.is_contiguous()
    return v, v.resolve_conj().resolve_neg().clone(), r, c


CASES = [("conj", torch.complex64), ("conj", torch.complex128), ("neg", torch.float32),
         ("neg", torch.float64)]


@pytest.mark.parametrize("kind,dtype", CASES, ids=str)
@pytest.mark.parametrize("nnz", [1, 5000])
def test_operators(kind, dtype, nnz):
    v, plain, r, c = _view(kind, nnz, dtype)
    x = torch.arange(1, N + 1, device=DEV).to(dtype)
    B = torch.stack([x, -x, x], 1)
    for op in ("non", "trans", "conj"):
        assert torch.equal(flagsparse_spmv_coo(v, r, c, x, (N, N), op=op),
                           flagsparse_spmv_coo(plain, r, c, x, (N, N), op=op))
    dense = torch.zeros((N, N), dtype=torch.complex128, device=DEV)
    dense.index_put_((r, c), plain.to(torch.complex128), accumulate=True)
    want = dense @ B.to(torch.complex128)
    assert torch.equal(flagsparse_spmm_coo(v, r, c, B, (N, N)).to(torch.complex128), want)
    assert torch.equal(flagsparse_spmv_coo(v, r, c, x, (N, N)).to(torch.complex128), want[:, 0])


@pytest.mark.parametrize("kind,dtype", CASES, ids=str)
def test_sorted_values(kind, dtype):
    v, plain, r, c = _view(kind, 5000, dtype)
    p = prepare_spmv_coo(v, r, c, (N, N))
    assert torch.equal(p.data, prepare_spmv_coo(plain, r, c, (N, N)).data)
    d = coo_to_csr_for_spmv(v, r, c, (N, N))[0]
    assert torch.equal(d, coo_to_csr_for_spmv(plain, r, c, (N, N))[0])
    assert not d.is_conj() and not d.is_neg()
