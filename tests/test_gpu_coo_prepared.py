"""PreparedCoo as an object: copies, saved files, its run bounds and counts, arrays
set before the first product."""

import copy
import io

import numpy as np
import pytest
import torch

from flagsparse_public_amd import flagsparse_spmv_coo, prepare_spmv_coo

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
N, M, NNZ = 400, 300, 3000


def _entries():
    rng = np.random.default_rng(1)
    r, c = rng.integers(0, N, NNZ), rng.integers(0, M, NNZ)
    v = rng.integers(-4, 5, NNZ).astype(np.float64)
    dense = np.zeros((N, M))
    np.add.at(dense, (r, c), v)
    return [torch.from_numpy(a).to(DEV) for a in (v, r, c)], torch.from_numpy(dense).to(DEV), r


def _saved(p):
    f = io.BytesIO()
    torch.save(p, f)
    f.seek(0)
    return torch.load(f, weights_only=False)


@pytest.mark.parametrize("clone", [copy.copy, copy.deepcopy, _saved], ids=["copy", "deepcopy", "save"])
def test_clones(clone):
    args, dense, r = _entries()
    x = torch.arange(M, device=DEV, dtype=torch.float64)
    p = clone(prepare_spmv_coo(*args, (N, M)))
    assert torch.equal(flagsparse_spmv_coo(x=x, prepared=p), dense @ x)
    rs = np.sort(r)
    starts = np.concatenate([[0], np.nonzero(rs[1:] != rs[:-1])[0] + 1, [NNZ]])
    assert p.n_segs == starts.size - 1
    assert np.array_equal(p.seg_starts.cpu().numpy(), starts)


def test_n_segs_is_a_plain_number(monkeypatch):
    args, _, r = _entries()
    p = prepare_spmv_coo(*args, (N, M))
    monkeypatch.setattr(torch, "nonzero", None)  # what the bounds are built with
    assert p.n_segs == np.unique(r).size and p.use_seg_kernel
    p.n_segs = 5
    assert p.n_segs == 5
    assert prepare_spmv_coo(*args, (N, M), sort_by_row=False).n_segs == 0


def test_arrays_set_before_the_first_product():
    """A product takes the arrays that the object holds at that time."""
    args, dense, _ = _entries()
    x = torch.arange(M, device=DEV, dtype=torch.float64)
    other = torch.sort(torch.randint(0, N, (NNZ,), device=DEV)).values
    p = prepare_spmv_coo(*args, (N, M))
    p.row = other
    want = torch.zeros((N, M), dtype=torch.float64, device=DEV)
    want.index_put_((other, p.col), p.data, accumulate=True)
    assert torch.equal(flagsparse_spmv_coo(x=x, prepared=p), want @ x)
    p = prepare_spmv_coo(*args, (N, M))
    p.row.copy_(other)
    assert torch.equal(flagsparse_spmv_coo(x=x, prepared=p), want @ x)
    p = prepare_spmv_coo(*args, (N, M))
    p.data.mul_(2)  # values alone may change
    assert torch.equal(flagsparse_spmv_coo(x=x, prepared=p), 2 * (dense @ x))


def test_columns_set_before_the_first_product_are_checked():
    args, _, _ = _entries()
    x = torch.ones(M, device=DEV, dtype=torch.float64)
    p = prepare_spmv_coo(*args, (N, M))
    p.col[7] = M
    with pytest.raises(IndexError):
        flagsparse_spmv_coo(x=x, prepared=p)
