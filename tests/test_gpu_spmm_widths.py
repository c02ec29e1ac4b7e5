"""SpMM lane shapes: every value type at dense widths around the edges of the
lane segments (16 bytes per lane) and lane groups, with B and C rows that
start at any element (odd leading dimensions, offset bases), against the fp64
oracle.

Bar per element, S = |A| |B|, C0 the old C: fp64 sums of fp32 values round
once (2^-24 |C| with slack for the fp64 sum), fp32 sums of 16-bit values err
by at most (len + 2) 2^-24 S before the rounding to the stored type
(2^-11 |C| fp16, 2^-8 |C| bf16), fp64 / complex by (len + 4) units of their
precision times S (complex: two products per component, factor 4)."""

import numpy as np
import pytest
import torch

from tests._util import to_dev

pytestmark = pytest.mark.gpu

from flagsparse_public_amd import _lib, flagsparse_spmm_csr  # noqa: E402
from flagsparse_public_amd.rowsplit import RowSplitPlan, Schedule  # noqa: E402

DTYPES = (torch.float16, torch.bfloat16, torch.float32, torch.float64, torch.complex32,
          torch.complex64, torch.complex128)
LENS = np.concatenate([np.arange(40), [0, 64, 65, 300, 1100], np.full(30, 7)])
M = 900


def _bar(dtype, C64, S, length):
    u = {torch.float64: 2.0**-53, torch.complex128: 2.0**-53}.get(dtype, 2.0**-24)
    out = {torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8, torch.complex32: 2.0**-11}.get(dtype, u)
    k = 4.0 if dtype.is_complex else 1.0
    tiny = 2.0**-24 if dtype in (torch.float16, torch.complex32) else 0.0  # fp16 subnormal step
    return k * (out * 1.01 * np.abs(C64) + (length[:, None] + 4.0) * u * S + tiny)


def _case(dtype, n_dense, seed):
    rng = np.random.default_rng(seed)
    ip = np.zeros(LENS.size + 1, np.int64)
    np.cumsum(LENS, out=ip[1:])
    cols = rng.integers(0, M, ip[-1]).astype(np.int32)

    def rand(shape):
        v = rng.uniform(-1, 1, shape)
        return v + 1j * rng.uniform(-1, 1, shape) if dtype.is_complex else v
    make = torch.complex64 if dtype == torch.complex32 else dtype
    vals = torch.from_numpy(rand(ip[-1])).to(make).to(dtype)
    B = torch.from_numpy(rand((M, n_dense))).to(make).to(dtype)
    C0 = torch.from_numpy(rand((LENS.size, n_dense))).to(make).to(dtype)
    return ip, cols, vals, B, C0


def _wide(t):
    return (t.to(torch.complex64) if t.dtype == torch.complex32 else t).to(
        torch.complex128 if t.dtype.is_complex else torch.float64).numpy()


def _place(t, ld, offset):
    """A device copy of the 2-D tensor t inside a larger buffer: leading
    dimension ld, first element `offset` elements past an aligned base."""
    n, m = t.shape
    buf = torch.zeros(offset + n * ld + 16, dtype=t.dtype, device="cuda")
    view = buf[offset:offset + n * ld].view(n, ld)[:, :m]
    view.copy_(t)
    return buf, view


@pytest.mark.parametrize("n_dense", [1, 7, 8, 9, 15, 16, 17, 31, 33, 47, 63, 65, 127, 129, 300])
@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).replace("torch.", ""))
def test_widths_strides_and_offsets(orc, dtype, n_dense):
    ip, cols, vals, B, C0 = _case(dtype, n_dense, n_dense)
    v64, B64, O64 = _wide(vals), _wide(B), _wide(C0)
    P64 = orc.spmm(ip, cols, v64, B64)
    S = orc.spmm_abs(ip, cols, v64, B64)
    acc = _lib.FS_ACC_WIDE if dtype == torch.float32 else _lib.FS_ACC_NATIVE
    ipd, cd, vd = to_dev(ip), to_dev(cols), vals.cuda()
    csr = _lib.make_csr(vd, cd, ipd, LENS.size, M)
    # long rows chunked (several chunks, one chunk) and none; padded and odd rows
    for k, (sch, pad, off) in enumerate([
            (Schedule(short_max=256, chunk_nnz=256), 0, 0),
            (Schedule(short_max=32, chunk_nnz=64), 1, 1),
            (Schedule(short_max=1 << 40, chunk_nnz=64, unroll=8), 3, 5),
            (Schedule(short_max=32, chunk_nnz=512, col_tile=20, unroll=8), 0, 3)]):
        plan = RowSplitPlan(ipd, LENS.size, dtype, sch, acc)
        _, Bv = _place(B, n_dense + pad, off)
        cbuf, Cv = _place(C0, n_dense + pad, off)
        beta = 0.0 if k % 2 == 0 else 0.5
        _lib.spmm(csr, Bv, n_dense + pad, Cv, n_dense + pad, n_dense, 1.0, beta,
                  plan.struct(n_dense), sch.col_tile, vd.device)
        want = P64 + beta * O64
        got = _wide(Cv.contiguous().cpu())
        bar = _bar(dtype, np.abs(P64) + beta * np.abs(O64), S + beta * np.abs(O64), LENS)
        assert np.all(np.abs(got - want) <= bar), (k, np.max(np.abs(got - want) / bar))
        # nothing outside the view is written
        keep = torch.ones(cbuf.numel(), dtype=torch.bool, device="cuda")
        keep[off:off + LENS.size * (n_dense + pad)].view(LENS.size, -1)[:, :n_dense] = False
        rest = torch.view_as_real(cbuf) if dtype.is_complex else cbuf
        assert torch.count_nonzero(rest[keep]).item() == 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.complex64], ids=["bf16", "c64"])
def test_special_values_stay_in_their_columns(dtype):
    """inf and NaN in one column of B reach that column of C only (the shifted
    tail window computes shared columns twice and writes them once)."""
    n_dense, tail = 37, 36
    B = torch.ones((4, n_dense), dtype=dtype, device="cuda")
    B[1, tail] = float("inf")
    B[2, 3] = float("nan")
    ip = torch.tensor([0, 2, 4], device="cuda")
    ci = torch.tensor([0, 1, 0, 2], dtype=torch.int32, device="cuda")
    data = torch.ones(4, dtype=dtype, device="cuda")
    C = torch.view_as_real(flagsparse_spmm_csr(data, ci, ip, B, (2, 4)).to(torch.complex64))
    bad = ~torch.isfinite(C).all(dim=2)
    assert torch.nonzero(bad).tolist() == [[0, tail], [1, 3]]
