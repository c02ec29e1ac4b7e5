"""fs_csr_analyze_split: the long-row lists it writes beside the statistics,
against numpy, and the unprepared SpMM call that runs on them."""

import ctypes

import numpy as np
import pytest
import torch

from tests._util import to_dev

pytestmark = pytest.mark.gpu

from flagsparse_public_amd import _lib, flagsparse_spmm_csr  # noqa: E402

DEV = torch.device("cuda", 0)


def _matrix(lens, idx, ptr, seed=0):
    rng = np.random.default_rng(seed)
    ip = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    cols = rng.integers(0, 1000, ip[-1])
    return ip, cols, torch.from_numpy(cols).to(idx).to(DEV), torch.from_numpy(ip).to(ptr).to(DEV)


CASES = {
    "none": np.full(200, 7),
    "all_one_chunk": np.full(500, 40),
    "lane_edges": np.where(np.arange(400) % 63 == 0, 33, 3),
    "several_chunks": np.concatenate([np.full(70, 129), [0, 5000, 64, 65, 128, 32, 33]]),
    "one_row": np.array([100_000]),
    "empty": np.zeros(0, np.int64),
    "many_blocks": np.where(np.arange(90_000) % 97 == 0, 200, 2),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("idx,ptr", [(torch.int32, torch.int32), (torch.int64, torch.int64),
                                     (torch.int64, torch.int32)], ids=["i32", "i64", "i64p32"])
def test_lists(name, idx, ptr):
    lens, short, chunk = CASES[name], 32, 64
    ip, cols, cd, pd = _matrix(lens, idx, ptr)
    vals = torch.zeros(cols.size, device=DEV)
    csr = _lib.make_csr(vals, cd, pd, lens.size, 1000)
    stats, rows, cptr, owner, n_long, n_chunks, narrow, _ = _lib.analyze_split(
        csr, DEV, short, chunk, idx == torch.int64)
    assert stats == _lib.analyze(csr, DEV)
    per = -(-lens // chunk)
    long = np.nonzero(lens > short)[0]
    assert n_long == long.size and n_chunks == int(per[long].sum())
    got = rows[:n_long].cpu().numpy()
    assert np.array_equal(np.sort(got), long)  # the order of the list is free
    bounds = cptr[:n_long + 1].cpu().numpy()
    assert bounds[0] == 0 and np.array_equal(np.diff(bounds), per[got])
    assert np.array_equal(owner[:n_chunks].cpu().numpy(), np.repeat(np.arange(n_long), per[got]))
    if idx == torch.int64:
        assert torch.equal(narrow.cpu(), torch.from_numpy(cols).to(torch.int32))
    else:
        assert narrow is None


def test_bad_pointers_stay_inside_the_lists():
    """Lengths far beyond the entries (row pointers not yet validated): the
    statistics report them and nothing is written past the capacities."""
    ip = np.array([0, 50, 10**12, 3, 900, 900 + 10**9], np.int64)
    cd = torch.zeros(64, dtype=torch.int32, device=DEV)
    pd, vals = to_dev(ip), torch.zeros(64, device=DEV)
    csr = _lib.make_csr(vals, cd, pd, ip.size - 1, 10)
    stats = torch.zeros(_lib.FS_STATS_LEN + 1, dtype=torch.int64, device=DEV)
    rows = torch.full((8,), -9, dtype=torch.int64, device=DEV)
    cptr = torch.full((8,), -9, dtype=torch.int64, device=DEV)
    owner = torch.full((16,), -9, dtype=torch.int32, device=DEV)
    rc = _lib.load().fs_csr_analyze_split(ctypes.byref(csr), stats.data_ptr(), 32, 64,
                                          rows.data_ptr(), cptr.data_ptr(), 1, owner.data_ptr(), 2,
                                          None, _lib.stream_handle(DEV))
    assert rc == _lib.FS_OK
    assert stats[2].item() == 1 and stats[1].item() != 64
    assert rows[1:].eq(-9).all() and cptr[2:].eq(-9).all() and owner[2:].eq(-9).all()
    with pytest.raises(ValueError):
        flagsparse_spmm_csr(vals, cd, pd, torch.zeros((10, 4), device=DEV), (ip.size - 1, 10))


@pytest.mark.parametrize("name", [n for n in CASES if n != "empty"])
@pytest.mark.parametrize("idx", [torch.int32, torch.int64])
@pytest.mark.parametrize("n_dense", [3, 40])
def test_unprepared_spmm_on_the_lists(orc, name, idx, n_dense):
    """Whole-number inputs: every sum is exact, so the call equals the oracle."""
    lens = CASES[name]
    ip, cols, cd, pd = _matrix(lens, idx, idx)
    rng = np.random.default_rng(1)
    vals = rng.integers(-4, 5, cols.size).astype(np.float32)
    B = rng.integers(-4, 5, (1000, n_dense)).astype(np.float32)
    want = orc.spmm(ip, cols.astype(np.int32), vals.astype(np.float64), B.astype(np.float64))
    for _ in range(2):
        C = flagsparse_spmm_csr(to_dev(vals), cd, pd, to_dev(B), (lens.size, 1000))
        assert np.array_equal(C.double().cpu().numpy(), want)


def test_argument_checks():
    lib = _lib.load()
    csr = _lib.make_csr(torch.zeros(4, device=DEV), torch.zeros(4, dtype=torch.int32, device=DEV),
                        torch.tensor([0, 4], device=DEV), 1, 4)
    buf = torch.zeros(64, dtype=torch.int64, device=DEV)

    def call(**kw):
        a = dict(A=ctypes.byref(csr), stats=buf.data_ptr(), short=32, chunk=64,
                 rows=buf.data_ptr(), cptr=buf.data_ptr(), cap=1, owner=buf.data_ptr(), capc=1)
        a.update(kw)
        return lib.fs_csr_analyze_split(*a.values(), None, _lib.stream_handle(DEV))
    for bad in (dict(short=0), dict(chunk=0), dict(chunk=65), dict(cap=-1), dict(capc=-1),
                dict(rows=None), dict(cptr=None), dict(owner=None), dict(stats=None), dict(A=None),
                dict(cap=1 << 31)):
        assert call(**bad) == _lib.FS_ERR_VALUE, bad
