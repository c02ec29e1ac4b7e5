"""A batch of more items than one launch holds (2^32 work-items, 256 to an item)."""

import pytest
import torch

from flagsparse_public_amd.batched import BatchedCsr

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def test_more_than_2_24_items():
    n = (1 << 24) + 5
    ptr = torch.arange(n + 1, device=DEV, dtype=torch.int32)
    cols = torch.arange(n, device=DEV, dtype=torch.int32) % 1000
    vals = (torch.arange(n, device=DEV) % 7 - 3).float()
    x = torch.arange(1, 1001, device=DEV).float()
    bat = BatchedCsr([dict(data=vals, indices=cols, indptr=ptr, shape=(n, 1000), x=x)], max_rows=1)
    assert bat.n_items == n
    bat.run()
    assert torch.equal(bat.y[0], vals * x[cols.long()])
