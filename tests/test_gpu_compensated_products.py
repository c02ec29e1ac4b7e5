"""Compensated fp32 sums over products that do not round to themselves: the sum's
correction holds each product's rounding once, so the result is the exact one,
rounded."""

import math
from fractions import Fraction

import numpy as np
import pytest
import torch

from flagsparse_public_amd import (flagsparse_spmm_csr_opt, flagsparse_spmv_csr,
                                   prepare_spmm_csr_opt, prepare_spmv_csr)
from flagsparse_public_amd.rowsplit import Schedule

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("n_dense", [0, 1, 8, 33, 64, 100])
def test_sums_are_the_exact_ones_rounded(n_dense):
    """Rows of 130 and 700 entries in chunks, factors of 24 random bits and both
    signs: sums of about 9, an ulp of 10^-6 apart.  The correction (up to about
    10^-5) rounds at 2^-24 of itself, 700 times: the result is off by an ulp where
    the exact value lies within some 10^-11 of the middle of two numbers, one in
    10^5.  The products' roundings counted twice are some 3 10^-7, one in five."""
    rng = np.random.default_rng(n_dense)
    lens = np.array([130, 700] * 40)
    ptr = np.concatenate([[0], np.cumsum(lens)])
    n_cols = 900
    cols = np.concatenate([rng.permutation(n_cols)[:n] for n in lens]).astype(np.int32)
    vals = (2 * rng.random(ptr[-1]) - 1).astype(np.float32)
    B = (2 * rng.random((n_cols, max(n_dense, 1))) - 1).astype(np.float32)
    f = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    sch = Schedule(group_lanes=8, short_max=32, chunk_nnz=256)
    args = (f(vals), f(cols), f(ptr), (lens.size, n_cols))
    if n_dense:
        got = flagsparse_spmm_csr_opt(B=f(B), prepared=prepare_spmm_csr_opt(*args, schedule=sch))
    else:
        got = flagsparse_spmv_csr(x=f(B[:, 0].copy()), use_opt=True,
                                  prepared=prepare_spmv_csr(*args, schedule=sch))[:, None]
    got = got.cpu().numpy()
    v64, B64 = vals.astype(np.float64), B.astype(np.float64)  # products of floats: exact
    wrong = 0
    for r in range(lens.size):
        prod = v64[ptr[r]:ptr[r + 1], None] * B64[cols[ptr[r]:ptr[r + 1]]]
        for n in range(got.shape[1]):
            # exact products; fractions in the first columns, fsum in the others: both exact
            exact = sum(map(Fraction, prod[:, n])) if n < 2 else math.fsum(prod[:, n])
            wrong += got[r, n] != np.float32(float(exact))
    assert wrong <= 0.005 * got.size
