"""coo_to_csr_for_spmv over the forms of its arguments that are plain torch
operations: value types, values with gradients, more values than index pairs."""

import numpy as np
import pytest
import torch

from flagsparse_public_amd import flagsparse_spmv_coo, prepare_spmv_coo
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


def test_gradients_reach_the_values():
    r, c, order = _pairs()
    data = torch.randn(NNZ, device=DEV, requires_grad=True)
    d, _, _ = coo_to_csr_for_spmv(data, r, c, (N, M))
    w = torch.randn(NNZ, device=DEV)
    (d * w).sum().backward()
    want = torch.empty_like(w)
    want[order] = w
    assert torch.equal(data.grad, want)
    with torch.no_grad():
        assert torch.equal(coo_to_csr_for_spmv(data, r, c, (N, M))[0], data[order])


def test_tangents_reach_the_values():
    import torch.autograd.forward_ad as fwd
    r, c, order = _pairs()
    data, t = torch.randn(NNZ, device=DEV), torch.randn(NNZ, device=DEV)
    with fwd.dual_level():
        d = coo_to_csr_for_spmv(fwd.make_dual(data, t), r, c, (N, M))[0]
        primal, tangent = fwd.unpack_dual(d)
        assert torch.equal(primal, data[order]) and torch.equal(tangent, t[order])


class _Marked(torch.Tensor):
    pass


def test_subclasses_stay():
    r, c, order = _pairs()
    data = torch.randn(NNZ, device=DEV)
    d = coo_to_csr_for_spmv(data.as_subclass(_Marked), r, c, (N, M))[0]
    assert type(d) is _Marked and torch.equal(d.as_subclass(torch.Tensor), data[order])


@pytest.mark.parametrize("shape", [(NNZ + 300,), (NNZ, 3), (NNZ + 5, 2)], ids=str)
def test_more_values_than_pairs(shape):
    """The values are indexed by the pairs' order whatever else they hold."""
    r, c, order = _pairs()
    data = torch.randn(shape, device=DEV)
    d, cols, ip = coo_to_csr_for_spmv(data, r, c, (N, M))
    assert torch.equal(d, data[order]) and torch.equal(cols, c[order].to(torch.int32))
    assert ip[-1].item() == NNZ


def test_function_transforms_reach_the_values():
    r, c, order = _pairs()
    w = torch.randn(NNZ, device=DEV)

    def f(v):
        return (coo_to_csr_for_spmv(v, r, c, (N, M))[0] * w).sum()
    data = torch.randn(3, NNZ, device=DEV)
    want = torch.empty_like(w)
    want[order] = w
    assert torch.equal(torch.func.grad(f)(data[0]), want)
    many = torch.vmap(lambda v: coo_to_csr_for_spmv(v, r, c, (N, M))[0])(data)
    assert torch.equal(many, data[:, order])


def test_prepared_values_keep_their_gradients():
    r, c, order = _pairs()
    data = torch.randn(NNZ, device=DEV, requires_grad=True)
    w = torch.randn(NNZ, device=DEV)
    want = torch.empty_like(w)
    want[order] = w
    p = prepare_spmv_coo(data, r, c, (N, M))
    (grad,) = torch.autograd.grad((p.data * w).sum(), data)
    assert torch.equal(grad, want)
    x = torch.randn(M, device=DEV)
    y = flagsparse_spmv_coo(x=x, prepared=p)
    assert torch.equal(y, flagsparse_spmv_coo(data, r, c, x, (N, M)))
    assert not y.requires_grad
