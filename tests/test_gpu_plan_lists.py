"""RowSplitPlan with and without the matrix size: the native listing of the long
rows against the torch operators' lists, for row pointers of both widths."""

import numpy as np
import pytest
import torch

from flagsparse_public_amd import _lib
from flagsparse_public_amd.rowsplit import RowSplitPlan, Schedule

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("ptr", [torch.int32, torch.int64])
@pytest.mark.parametrize("short,chunk", [(1, 64), (64, 64), (64, 512), (10_000, 256)])
@pytest.mark.parametrize("rows", [1, 63, 3000, 50_000])
def test_lists(rows, short, chunk, ptr):
    rng = np.random.default_rng(rows)
    lens = np.minimum(1.0 / (1.0 - rng.random(rows)), 9000).astype(np.int64) - 1
    lens[rows // 2] = 9000
    ip = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)])).to(ptr).to(DEV)
    sch = Schedule(group_lanes=8, short_max=short, chunk_nnz=chunk)
    want = RowSplitPlan(ip, rows, torch.float32, sch, _lib.FS_ACC_NATIVE)
    got = RowSplitPlan(ip, rows, torch.float32, sch, _lib.FS_ACC_NATIVE, nnz=int(lens.sum()))
    assert (got.n_long, got.n_chunks, got.n_tiles) == (want.n_long, want.n_chunks, 0)
    order = torch.argsort(got.long_rows)  # the order of the list is free
    assert torch.equal(got.long_rows[order], want.long_rows)
    if got.n_long:
        assert torch.equal(torch.diff(got.long_chunk_ptr)[order], torch.diff(want.long_chunk_ptr))
    owner = torch.repeat_interleave(torch.arange(got.n_long, device=DEV),
                                    torch.diff(got.long_chunk_ptr))
    assert torch.equal(got.chunk_long.to(torch.int64), owner)
