"""coo_to_csr_for_spmv over the forms of its arguments that are plain torch
operations: value types, values with gradients, more values than index pairs."""

import numpy as np
import pytest
import torch

from flagsparse_public_amd.sparse_operations.spmv_csr import coo_to_csr_for_spmv

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
N, M, NNZ = 60, 50, 700


def _pairs():
    rng = np.random.default_rng(2)
    r, c = rng.integers(0, N, NNZ), rng.integers(0, M, NNZ)
    order = torch.from_numpy(np.lexsort((np.arange(NNZ), c, r))).to(DEV)
    return torch.from_numpy(r).to(DEV), torch.from_numpy(c).to(DEV), order


@pytest.mark.parametrize("dtype", [torch.bool, torch.uint8, torch.int8, torch.int16, torch.float16,
                                   torch.bfloat16, torch.float32, torch.int64, torch.complex128],
                         ids=str)
def test_value_types(dtype):
    r, c, order = _pairs()
    data = (torch.arange(NNZ, device=DEV) % 101).to(dtype)
    d, cols, _ = coo_to_csr_for_spmv(data, r, c, (N, M))
    assert torch.equal(d, data[order]) and torch.equal(cols, c[order].to(torch.int32))


@pytest.mark.parametrize("shape", [(NNZ + 300,), (NNZ, 3), (NNZ + 5, 2)], ids=str)
def test_more_values_than_pairs(shape):
    """The values are indexed by the pairs' order whatever else they hold."""
    r, c, order = _pairs()
    data = torch.randn(shape, device=DEV)
    d, cols, ip = coo_to_csr_for_spmv(data, r, c, (N, M))
    assert torch.equal(d, data[order]) and torch.equal(cols, c[order].to(torch.int32))
    assert ip[-1].item() == NNZ
