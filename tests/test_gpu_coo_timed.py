"""What a timed COO SpMM times: the sort and the product, behind the checks of the
arrays and, where those are passes of their own, of the indices."""

import pytest
import torch

from flagsparse_public_amd import flagsparse_spmm_coo
from flagsparse_public_amd.sparse_operations import spmm_coo

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("native", [True, False])
def test_the_clock_starts_behind_the_checks(native, monkeypatch):
    seen = []

    def note(module, name, mark):
        was = getattr(module, name)
        monkeypatch.setattr(module, name, lambda *a, **k: (seen.append(mark), was(*a, **k))[1])
    note(spmm_coo, "_check_spmm_coo_arrays", "arrays")
    note(spmm_coo, "_prepare_spmm_coo_inputs", "indices")
    note(spmm_coo.time, "perf_counter", "clock")
    if not native:
        monkeypatch.setattr(spmm_coo._lib, "coo_sort_applies", lambda *a: False)
    r, c = torch.randint(0, 40, (900,), device=DEV), torch.randint(0, 30, (900,), device=DEV)
    v = torch.randint(-3, 4, (900,), device=DEV).double()
    B = torch.randint(-3, 4, (30, 5), device=DEV).double()
    C, ms = flagsparse_spmm_coo(v, r, c, B, (40, 30), return_time=True)
    dense = torch.zeros((40, 30), dtype=torch.float64, device=DEV)
    dense.index_put_((r, c), v, accumulate=True)
    assert torch.equal(C, dense @ B) and ms > 0
    assert seen.index("arrays") < seen.index("clock")
    if native:
        assert seen == ["arrays", "clock", "clock"]
    else:
        last = len(seen) - 1
        assert seen[-2:] == ["clock", "clock"] and "indices" in seen[:last - 1]
