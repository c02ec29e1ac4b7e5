"""BatchedCsr over widths, alignments and row counts at the edges of its items:
whole-number inputs whose sums are exact, so results must equal the integers."""

import numpy as np
import pytest
import torch

from flagsparse_public_amd import _lib
from flagsparse_public_amd.batched import BatchedCsr

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _matrix(rng, rows, n_cols, mean, n_dense, lanes, offset):
    lens = rng.integers(0, 2 * mean + 1, rows)
    if rows > 40:
        lens[rows // 2] = 5000  # above long_row, and a range above item_bytes
    ip = np.concatenate([[0], np.cumsum(lens)])
    cols, vals = rng.integers(0, n_cols, ip[-1]), rng.integers(-2, 3, ip[-1])
    x, B = rng.integers(-2, 3, n_cols), rng.integers(-2, 3, (n_cols, n_dense))
    P = np.zeros((rows, n_cols), np.int64)
    np.add.at(P, (np.repeat(np.arange(rows), lens), cols), vals)
    buf = torch.zeros(n_cols * n_dense + offset, device=DEV)  # B at an odd address
    buf[offset:] = torch.from_numpy(B).to(torch.float32).flatten().to(DEV)
    f = lambda a, t: torch.from_numpy(np.ascontiguousarray(a)).to(t).to(DEV)  # noqa: E731
    d = {"data": f(vals, torch.float32), "indices": f(cols, torch.int32),
         "indptr": f(ip, torch.int32 if offset else torch.int64), "shape": (rows, n_cols),
         "x": f(x, torch.float32), "B": buf[offset:].view(n_cols, n_dense), "group_lanes": lanes}
    return d, P @ x, P @ B


@pytest.mark.parametrize("n_dense", [1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 31, 32, 33, 64, 65, 130, 260, 300])
@pytest.mark.parametrize("item_bytes", [96 * 1024, 1000])
def test_widths_and_edges(n_dense, item_bytes):
    rng = np.random.default_rng(n_dense)
    rows = _lib.load().fs_batch_rows(8, n_dense)
    mats, ys, Cs = zip(*[_matrix(rng, r, 97, m, n_dense, lanes, off) for r, m, lanes, off in (
        (1, 3, 1, 0), (rows, 6, 8, 1), (rows + 1, 6, 64, 2), (2 * rows - 1, 2, 2, 3), (300, 9, 32, 0))])
    b = BatchedCsr(list(mats), item_bytes=item_bytes)
    for alpha, beta in ((1.0, 0.0), (2.0, 3.0)):
        before = [(y.clone(), C.clone()) for y, C in zip(b.y, b.C)]
        b.run(alpha, beta)
        for k, (y0, C0) in enumerate(before):
            assert np.array_equal(b.y[k].cpu().numpy(), alpha * ys[k] + beta * y0.cpu().numpy())
            assert np.array_equal(b.C[k].cpu().numpy(), alpha * Cs[k] + beta * C0.cpu().numpy())


def test_rows_of_an_item():
    f = _lib.load().fs_batch_rows
    assert [f(s, 0) for s in (1, 8, 32, 64)] == [1024, 128, 32, 16]
    assert [f(8, n) for n in (1, 4, 8, 16, 32, 64, 128, 256, 1000)] == [64, 64, 32, 32, 32, 16, 8, 4, 4]
