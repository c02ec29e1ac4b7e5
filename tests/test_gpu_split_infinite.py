"""Split-precision SpMV with an infinite x: the rows that meet it are infinite (their
compensated sums' correction alone would make them NaN), the others are exact, in
every role that sums a row: lane groups, chunks, entry tiles, column slices, windows."""

import numpy as np
import pytest
import torch

from flagsparse_public_amd.precision import flagsparse_spmv_csr_split, prepare_spmv_csr_split
from flagsparse_public_amd.rowsplit import Schedule

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
N_COLS = 9000
LENGTHS = (1, 20, 300, 3000, 9000)


@pytest.mark.parametrize("fmt", ["bf16x2", "bf16", "f16_rowscale"])
@pytest.mark.parametrize("sch", [
    None,
    Schedule(group_lanes=4, short_max=64, chunk_nnz=512, unroll=4),
    Schedule(tile_nnz=2048, tile_mode=1),
    Schedule(tile_nnz=4096, tile_mode=1),
    Schedule(tile_nnz=2048, tile_mode=1, x_slice_cols=4096),
    Schedule(group_lanes=8, short_max=2048, chunk_nnz=8192, unroll=4, tile_nnz=2048),
    Schedule(tile_nnz=2048, tile_mode=1, x_window=1024),
])
@pytest.mark.parametrize("special", [float("inf"), -float("inf")])
def test_rows_that_meet_an_infinity(fmt, sch, special):
    """Ones in columns that hold 1, and every second row the last column, which
    holds the infinity; sums of at most 9,000 ones (exact)."""
    lens = np.array([n for n in LENGTHS for _ in range(2)] + [1, 20] * 400)
    meets = np.arange(lens.size) % 2 == 1
    cols = [np.arange(n) % (N_COLS - 1) for n in lens]
    for r in np.flatnonzero(meets):
        cols[r][-1] = N_COLS - 1
    cols = np.concatenate([np.sort(c) for c in cols]).astype(np.int32)
    ptr = np.concatenate([[0], np.cumsum(lens)])
    x = np.ones(N_COLS, np.float32)
    x[-1] = special
    f = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    p = prepare_spmv_csr_split(f(np.ones(ptr[-1], np.float32)), f(cols), f(ptr),
                               (lens.size, N_COLS), fmt, schedule=sch)
    y = flagsparse_spmv_csr_split(f(x), p).cpu().numpy()
    np.testing.assert_array_equal(y, np.where(meets, np.float32(special), lens.astype(np.float32)))
