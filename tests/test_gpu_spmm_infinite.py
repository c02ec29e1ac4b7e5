"""SpMM rows with infinities and sums that overflow: the result itself (+-inf, or
NaN where the exact sum has none), in rows of one lane group, in rows of one chunk
and in rows of several."""

import pytest
import torch

from flagsparse_public_amd import (flagsparse_spmm_coo, flagsparse_spmm_csr,
                                   flagsparse_spmm_csr_opt, prepare_spmm_csr_opt)
from flagsparse_public_amd.rowsplit import Schedule

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
INF = float("inf")
N_COLS, N_DENSE = 700, 21
# entries of a row: short, one chunk, several chunks (and more per fix-up lane)
LENGTHS = (20, 100, 200, 256, 300, 700)


def _matrix(dtype, what):
    """Rows of ones; `what` is set at two places of every second row.  The empty
    rows keep the mean length low."""
    lens = [n for n in LENGTHS for _ in range(2)] + [0] * 2000
    data, cols, ptr = [], [], [0]
    for i, n in enumerate(lens):
        row = torch.ones(n, dtype=torch.float64)
        if i % 2 and n:
            row[n // 3], row[n - 2] = what
        data.append(row)
        cols.append(torch.arange(n))
        ptr.append(ptr[-1] + n)
    return (torch.cat(data).to(dtype).to(DEV), torch.cat(cols).to(torch.int32).to(DEV),
            torch.tensor(ptr).to(DEV), len(lens))


def _check(C, plain, special):
    C = C[:2 * len(LENGTHS)].double().cpu()
    n = torch.tensor(LENGTHS, dtype=torch.float64)
    want = (n[:, None] * plain).expand(-1, N_DENSE).clone()
    assert torch.equal(C[0::2], want)  # <= 256 in bfloat16, 700 in the others: exact
    want[:] = special
    got = C[1::2]
    assert torch.equal(got.nan_to_num(nan=7.0), want.nan_to_num(nan=7.0))


def _call(kind, data, cols, ptr, n_rows, B):
    shape = (n_rows, N_COLS)
    if kind == "csr":
        return flagsparse_spmm_csr(data, cols, ptr, B, shape)
    if kind == "coo":
        rows = torch.repeat_interleave(torch.arange(n_rows, device=DEV), ptr[1:] - ptr[:-1])
        order = torch.randperm(rows.numel(), device=DEV)
        return flagsparse_spmm_coo(data[order], rows[order], cols.long()[order], B, shape)
    sch = Schedule(group_lanes=1, short_max=32, chunk_nnz=128) if kind == "given" else None
    return flagsparse_spmm_csr_opt(B=B, prepared=prepare_spmm_csr_opt(data, cols, ptr, shape,
                                                                     schedule=sch))


KINDS = [("csr", torch.float16), ("csr", torch.bfloat16), ("csr", torch.float32),
         ("csr", torch.float64), ("coo", torch.float16), ("coo", torch.bfloat16),
         ("coo", torch.float32), ("opt", torch.float32), ("opt", torch.float64),
         ("given", torch.float32)]


@pytest.mark.parametrize("kind,dtype", KINDS, ids=str)
@pytest.mark.parametrize("what,special", [((INF, 1.0), INF), ((-INF, 1.0), -INF),
                                          ((INF, INF), INF), ((INF, -INF), float("nan")),
                                          ((float("nan"), 1.0), float("nan"))], ids=str)
def test_entries(kind, dtype, what, special):
    data, cols, ptr, n_rows = _matrix(dtype, what)
    # ones in bfloat16 sum to 300 and 700 only after rounding: halves, quarters
    scale = 0.25 if dtype == torch.bfloat16 else 1.0
    B = torch.full((N_COLS, N_DENSE), scale, dtype=dtype, device=DEV)
    _check(_call(kind, data, cols, ptr, n_rows, B), scale, special)


@pytest.mark.parametrize("kind,dtype", [("opt", torch.float32), ("given", torch.float32),
                                        ("csr", torch.bfloat16), ("coo", torch.bfloat16)], ids=str)
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_sums_that_overflow(kind, dtype, sign):
    """Two of the largest finite products: their sum overflows fp32."""
    big = torch.finfo(dtype).max * sign
    data, cols, ptr, n_rows = _matrix(dtype, (big, big))
    scale = 0.25 if dtype == torch.bfloat16 else 1.0
    B = torch.full((N_COLS, N_DENSE), scale, dtype=dtype, device=DEV)
    if dtype == torch.bfloat16:
        # every entry's column is its place in the row: make the two products whole
        for n in LENGTHS:
            B[n // 3], B[n - 2] = 1.0, 1.0
        C = _call(kind, data, cols, ptr, n_rows, B)[:2 * len(LENGTHS)]
        assert bool((C[1::2].double() == sign * INF).all())
        assert bool(torch.isfinite(C[0::2]).all())
        return
    _check(_call(kind, data, cols, ptr, n_rows, B), scale, sign * INF)
