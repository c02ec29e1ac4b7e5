"""Prepared SpMM over several dense widths: the plans of all widths are there after
the first product, so that a product with another width can be recorded into a graph
and reads nothing back."""

import numpy as np
import pytest
import torch

from flagsparse_public_amd import (flagsparse_spmm_csr_opt, flagsparse_spmm_csr_opt_alg2,
                                   prepare_spmm_csr_opt, prepare_spmm_csr_opt_alg2)

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
WIDTHS = (1, 8, 33, 64, 65, 128, 200, 260)
RUN = {"opt": (prepare_spmm_csr_opt, flagsparse_spmm_csr_opt),
       "alg2": (prepare_spmm_csr_opt_alg2, flagsparse_spmm_csr_opt_alg2)}


def _matrix(n_rows, length, dtype, long_rows=5):
    rng = np.random.default_rng(n_rows)
    lens = rng.integers(0, 2 * length + 1, n_rows)
    lens[rng.permutation(n_rows)[:long_rows]] = 1500
    ptr = np.concatenate([[0], np.cumsum(lens)])
    cols = rng.integers(0, 700, ptr[-1]).astype(np.int32)
    vals = rng.integers(-2, 3, ptr[-1]).astype(np.float64)  # whole numbers: exact results
    dense = np.zeros((n_rows, 700))
    np.add.at(dense, (np.repeat(np.arange(n_rows), lens), cols), vals)
    f = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    return f(vals).to(dtype), f(cols), f(ptr), (n_rows, 700), f(dense)


@pytest.mark.parametrize("which", ["opt", "alg2"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=str)
@pytest.mark.parametrize("n_rows,length", [(3000, 10), (2000, 90), (900, 300)])
@pytest.mark.parametrize("first", [1, 260])
def test_one_width_plans_all(which, dtype, n_rows, length, first, monkeypatch):
    data, cols, ptr, shape, dense = _matrix(n_rows, length, dtype)
    prepare, run = RUN[which]
    p = prepare(data, cols, ptr, shape)
    B = {n: torch.randint(-2, 3, (shape[1], n), device=DEV).to(dtype) for n in WIDTHS}
    run(B=B[first], prepared=p)
    reads = []
    for name in ("cpu", "item", "tolist"):
        was = getattr(torch.Tensor, name)
        monkeypatch.setattr(torch.Tensor, name,
                            lambda t, *a, was=was, **k: (reads.append(name), was(t, *a, **k))[1])
    got = {n: run(B=B[n], prepared=p) for n in WIDTHS}
    monkeypatch.undo()
    assert not reads
    for n in WIDTHS:
        assert torch.equal(got[n].double(), dense @ B[n].double())


@pytest.mark.parametrize("which", ["opt", "alg2"])
def test_capture_of_another_width(which):
    data, cols, ptr, shape, dense = _matrix(3000, 10, torch.float32)
    prepare, run = RUN[which]
    p = prepare(data, cols, ptr, shape)
    run(B=torch.ones((shape[1], 8), device=DEV), prepared=p)  # the only width warmed
    for n in (64, 128, 260):
        B = torch.zeros((shape[1], n), device=DEV)
        out = torch.empty((shape[0], n), device=DEV)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            run(B=B, prepared=p, out=out)
        for i in range(3):
            B.copy_(torch.randint(-2, 3, B.shape, device=DEV))
            g.replay()
            eager = run(B=B, prepared=p)
            torch.cuda.synchronize()
            assert torch.equal(out.double(), dense @ B.double()) and torch.equal(out, eager)
