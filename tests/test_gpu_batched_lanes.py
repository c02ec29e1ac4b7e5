"""Lane counts that the batch refuses: the same error whatever the count."""

import pytest
import torch

from flagsparse_public_amd.batched import BatchedCsr, _lib_batch


@pytest.mark.parametrize("lanes", [-4, 3, 65, 256, 512, 1025, 1 << 20])
def test_rows_of_an_item_are_positive(lanes):
    assert _lib_batch().fs_batch_rows(lanes, 0) >= 1


@pytest.mark.gpu
@pytest.mark.parametrize("lanes", [-4, 3, 65, 512, 1025, 1 << 20])
def test_refused(lanes):
    f = lambda a, t: torch.tensor(a, dtype=t, device="cuda")  # noqa: E731
    m = dict(data=f([1.0], torch.float32), indices=f([0], torch.int32),
             indptr=f([0, 1], torch.int32), shape=(1, 1), x=f([1.0], torch.float32),
             group_lanes=lanes)
    with pytest.raises(ValueError, match="group_lanes must be a power of two"):
        BatchedCsr([m])
