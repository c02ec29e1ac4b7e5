"""SpMM launches of more blocks than one launch holds (2^32 work-items, 256 to a
block): 32 rows to a block here, with long rows at both ends and in the middle."""

import pytest
import torch

from flagsparse_public_amd import flagsparse_spmm_csr

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def test_more_than_2_24_blocks():
    n_rows, n_dense = (1 << 24) * 32 - 64, 8  # 2^24 - 2 blocks of rows, and those of chunks
    B = torch.randint(-1, 2, (700, n_dense), device=DEV).to(torch.bfloat16)
    rows = torch.tensor([0, 1, 31, n_rows // 2, n_rows - 33, n_rows - 1], device=DEV)
    lens = torch.tensor([200, 60, 40, 100, 200, 90], device=DEV)  # six chunks
    ptr = torch.zeros(n_rows + 1, dtype=torch.int32, device=DEV)
    ptr[rows + 1] = lens.int()
    ptr = torch.cumsum(ptr, 0, dtype=torch.int32)
    cols = torch.cat([torch.arange(n, device=DEV) for n in lens.tolist()]).int()
    data = (torch.arange(cols.numel(), device=DEV) % 3 - 1).to(torch.bfloat16)
    C = flagsparse_spmm_csr(data, cols, ptr, B, (n_rows, 700))
    prod = data.double()[:, None] * B.double()[cols.long()]
    want = torch.stack([p.sum(0) for p in prod.split(lens.tolist())])
    assert torch.equal(C[rows].double(), want)  # |sums| < 256: exact in bfloat16
    C[rows] = 0
    assert C.view(torch.int16).count_nonzero().item() == 0
