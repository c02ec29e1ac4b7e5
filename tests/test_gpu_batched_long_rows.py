"""Batched SpMM rows around the length where a whole block takes them, and far
beyond, in every lane group and column width; whole numbers, exact results."""

import numpy as np
import pytest
import torch

from flagsparse_public_amd import _lib
from flagsparse_public_amd.batched import BatchedCsr

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
LONG = _lib.FS_BATCH_LONG_MM
LENS = (3, LONG - 1, LONG, LONG + 1, 0, 1000, LONG + 1, 7, 5000, 20_003, 2)


def _matrix(n_dense, seed, index=torch.int32):
    rng = np.random.default_rng(seed)
    n_cols, lens = 400, np.array(LENS)
    ptr = np.concatenate([[0], np.cumsum(lens)])
    cols, vals = rng.integers(0, n_cols, ptr[-1]), rng.integers(-2, 3, ptr[-1])
    A = np.zeros((lens.size, n_cols))
    np.add.at(A, (np.repeat(np.arange(lens.size), lens), cols), vals)
    B = rng.integers(-2, 3, (n_cols, n_dense)).astype(np.float64)
    f = lambda a, t: torch.from_numpy(a).to(t).to(DEV)  # noqa: E731
    m = dict(data=f(vals, torch.float32), indices=f(cols, torch.int32), indptr=f(ptr, index),
             shape=A.shape, B=f(B, torch.float32), x=f(B[:, 0].copy(), torch.float32))
    return m, A @ B


@pytest.mark.parametrize("n_dense", [1, 3, 4, 5, 8, 9, 16, 17, 31, 32, 33, 64, 100, 129, 256, 257, 600])
@pytest.mark.parametrize("validate", [True, False])
def test_long_rows(n_dense, validate):
    ms, want = zip(*(_matrix(n_dense, s, t) for s, t in ((1, torch.int32), (2, torch.int64))))
    bat = BatchedCsr(list(ms), validate=validate)
    bat.run()
    for C, y, w in zip(bat.C, bat.y, want):
        assert np.array_equal(C.double().cpu().numpy(), w)
        assert np.array_equal(y.double().cpu().numpy(), w[:, 0])
    bat.run(alpha=2.0, beta=-1.0)
    for C, w in zip(bat.C, want):
        assert np.array_equal(C.double().cpu().numpy(), w)
    g = bat.capture()
    for _ in range(3):
        for C in bat.C:
            C.fill_(7.0)
        g.replay()
        torch.cuda.synchronize()
        for C, w in zip(bat.C, want):
            assert np.array_equal(C.double().cpu().numpy(), w)


def test_infinities_stay():
    m, want = _matrix(9, 3)
    row = 9  # the longest
    at = int(m["indptr"][row]) + 11_111
    m["data"][at] = float("inf")
    m["B"][m["indices"][at]] = 1.0
    bat = BatchedCsr([m])
    bat.run()
    assert bool((bat.C[0][row] == float("inf")).all())
    assert bool(torch.isfinite(bat.C[0][:row]).all())
