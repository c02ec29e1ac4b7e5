"""The SpMM's second pass over rows cut into chunks: chunk counts around the
edges of its lane ranges (1 chunk, up to 16 per way, one more, hundreds), dense
widths that give 64 to 1 ways per wavefront and several column tiles, alpha and
beta.

Values and B are whole numbers of at most 8, so every product, partial sum and
result is exact in fp32 whatever the order (below 2^23 quarters): the result
equals the fp64 oracle's bit for bit."""

import numpy as np
import pytest
import torch

from tests._util import to_dev

pytestmark = pytest.mark.gpu

from flagsparse_public_amd import _lib  # noqa: E402
from flagsparse_public_amd.rowsplit import RowSplitPlan, Schedule  # noqa: E402

CHUNK = 64
CHUNKS = (0, 1, 2, 15, 16, 17, 31, 33, 64, 65, 129, 300, 1, 1025, 3)


@pytest.mark.parametrize("n_dense", [1, 2, 3, 8, 31, 47, 64, 65, 130])
@pytest.mark.parametrize("mode", ["f32", "f32wide", "f64", "c64", "bf16"])
def test_chunk_counts(orc, mode, n_dense):
    rng = np.random.default_rng(n_dense)
    lens = np.array([max(0, c * CHUNK - int(rng.integers(0, CHUNK))) for c in CHUNKS] + [5, 9])
    ip = np.zeros(lens.size + 1, np.int64)
    np.cumsum(lens, out=ip[1:])
    m = 700
    dtype = {"f64": torch.float64, "c64": torch.complex64, "bf16": torch.bfloat16}.get(
        mode, torch.float32)

    def whole(shape):
        v = rng.integers(-8, 9, shape).astype(np.float64)
        return v + 1j * rng.integers(-8, 9, shape) if mode == "c64" else v
    cols = rng.integers(0, m, ip[-1]).astype(np.int32)
    vals, B, C0 = whole(ip[-1]), whole((m, n_dense)), whole((lens.size, n_dense))
    alpha, beta = 0.5, -0.25
    want = torch.from_numpy(alpha * orc.spmm(ip, cols, vals, B) + beta * C0).to(dtype)
    acc = _lib.FS_ACC_WIDE if mode == "f32wide" else _lib.FS_ACC_NATIVE
    ipd, cd, vd, Bd = to_dev(ip), to_dev(cols), to_dev(vals, dtype), to_dev(B, dtype)
    plan = RowSplitPlan(ipd, lens.size, dtype, Schedule(short_max=8, chunk_nnz=CHUNK), acc)
    csr = _lib.make_csr(vd, cd, ipd, lens.size, m)
    for _ in range(2):
        C = to_dev(C0, dtype)
        _lib.spmm(csr, Bd, n_dense, C, n_dense, n_dense, alpha, beta, plan.struct(n_dense), 0,
                  vd.device)
        assert torch.equal(C.cpu(), want)
