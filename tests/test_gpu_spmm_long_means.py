"""Precision of SpMM where rows are long on average: values far apart, of which a
plain fp32 sum of a row loses the small ones.  A compensated sum is exact and its
result fits every type, so nothing is left to a tolerance."""

import pytest
import torch

from flagsparse_public_amd import (flagsparse_spmm_coo, flagsparse_spmm_csr,
                                   flagsparse_spmm_csr_opt, prepare_spmm_csr_opt)

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("kind,dtype", [("csr", torch.float16), ("csr", torch.bfloat16),
                                        ("coo", torch.float16), ("coo", torch.bfloat16),
                                        ("opt", torch.float32)], ids=str)
@pytest.mark.parametrize("length,n_rows,n_dense", [(300, 4100, 256), (600, 4100, 256),
                                                   (1024, 4100, 256), (300, 33_000, 24)])
def test_small_values_are_kept(kind, dtype, length, n_rows, n_dense):
    last = length - 10
    data = torch.zeros(length, dtype=torch.float64)
    data[5], data[last] = 2.0**15, -(2.0**15)  # cancel
    # a quarter of an fp32 ulp of 2^15 each, few enough for bfloat16's 8 bits
    data[6:last:2][:128] = 2.0**-10
    want = data.sum().item()
    data = data.to(dtype).repeat(n_rows).to(DEV)
    cols = torch.arange(length, dtype=torch.int32, device=DEV).repeat(n_rows)
    ptr = torch.arange(n_rows + 1, device=DEV) * length
    B = torch.ones((length, n_dense), dtype=dtype, device=DEV)
    shape = (n_rows, length)
    if kind == "coo":
        rows = torch.repeat_interleave(torch.arange(n_rows, device=DEV), length)
        order = torch.randperm(rows.numel(), device=DEV)
        C = flagsparse_spmm_coo(data[order], rows[order], cols.long()[order], B, shape)
    elif kind == "csr":
        C = flagsparse_spmm_csr(data, cols, ptr, B, shape)
    else:
        p = prepare_spmm_csr_opt(data, cols, ptr, shape)
        C = flagsparse_spmm_csr_opt(B=B, prepared=p)
    assert bool((C.double() == want).all())
