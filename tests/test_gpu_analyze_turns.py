"""fs_csr_analyze_split over several turns of a block, with and without long
rows in them: the lists against numpy."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from flagsparse_public_amd import _lib  # noqa: E402

DEV = torch.device("cuda", 0)
TURN = 4 * 1024  # rows of one block and turn


@pytest.mark.parametrize("at", [(), (0,), (1, 3), (0, 1, 2, 3)], ids=str)
@pytest.mark.parametrize("rows", [4 * TURN, 4 * TURN - 1, 3 * TURN + 1])
def test_turns(rows, at):
    lens = np.zeros(rows, np.int64)  # few entries: one block walks all rows
    for k in at:
        lens[k * TURN:k * TURN + 200:67] = 70  # several wavefronts of the turn
        lens[min((k + 1) * TURN, rows) - 1] = 200
    ip = np.concatenate([[0], np.cumsum(lens)])
    nnz = int(ip[-1])
    assert max(rows, nnz) <= 1024 * 32
    cols = torch.zeros(nnz, dtype=torch.int32, device=DEV)
    vals, ptr = torch.zeros(nnz, device=DEV), torch.from_numpy(ip).to(torch.int32).to(DEV)
    csr = _lib.make_csr(vals, cols, ptr, rows, 1)
    stats, listed, cptr, owner, n_long, n_chunks, _, _ = _lib.analyze_split(csr, DEV, 32, 64, False)
    assert stats == _lib.analyze(csr, DEV)
    long = np.nonzero(lens > 32)[0]
    per = -(-lens // 64)
    got = listed[:n_long].cpu().numpy()
    assert np.array_equal(np.sort(got), long)
    bounds = cptr[:n_long + 1].cpu().numpy()
    assert n_chunks == int(per[long].sum()) and np.array_equal(np.diff(bounds), per[got])
    assert np.array_equal(owner[:n_chunks].cpu().numpy(), np.repeat(np.arange(n_long), per[got]))
