"""SDDMM over all row widths up to 70 and the edges above, with x and y at odd
addresses: whole-number inputs whose sums are exact, and values above the row's
end that must not be read into a sum."""

import numpy as np
import pytest
import torch

from flagsparse_public_amd import _lib

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("k", list(range(0, 71)) + [95, 96, 97, 127, 128, 129, 130, 131, 159, 160,
                                                    255, 256, 257, 258, 259, 511, 513])
@pytest.mark.parametrize("dtype,wide", [(torch.float32, False), (torch.float32, True),
                                        (torch.float64, False)], ids=["f32", "f32wide", "f64"])
def test_widths(k, dtype, wide):
    rng = np.random.default_rng(k)
    n, m, nnz = 37, 41, 301
    rows, cols = np.sort(rng.integers(0, n, nnz)), rng.integers(0, m, nnz)
    X, Y, D = rng.integers(-3, 4, (n, k)), rng.integers(-3, 4, (m, k)), rng.integers(-3, 4, nnz)

    def operand(a, off):  # off elements into its buffer, infinities around it
        buf = torch.full((a.size + off + 8,), float("inf"), dtype=dtype, device=DEV)
        buf[off:off + a.size] = torch.from_numpy(a).flatten().to(dtype).to(DEV)
        return buf[off:off + a.size]

    ip = torch.from_numpy(np.searchsorted(rows, np.arange(n + 1))).to(torch.int32).to(DEV)
    rid, cid = (torch.from_numpy(a).to(torch.int32).to(DEV) for a in (rows, cols))
    data, x, y = operand(D, 0), operand(X, k % 4), operand(Y, k % 3)
    csr = _lib.make_csr(data, cid, ip, n, m)
    for with_data in (True, False):
        if not with_data:
            csr.values = None
        out = torch.full((nnz,), 7.0, dtype=dtype, device=DEV)
        _lib.sddmm(csr, rid, x, y, k, out, csr.value_type,
                   _lib.FS_ACC_WIDE if wide else _lib.FS_ACC_NATIVE, 2.0, 3.0, DEV)
        want = 2 * (X[rows] * Y[cols]).sum(1) + 3 * with_data * D
        assert np.array_equal(out.cpu().numpy(), want.astype(np.float64))
