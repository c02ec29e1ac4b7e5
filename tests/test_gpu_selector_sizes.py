"""fs_mlp_select with networks on both sides of its LDS staging limit (12,288
parameters) and layers wider than a wavefront: scores equal the oracle's
forward pass, whose fp64 layer sums the kernel rounds to fp32 per layer (bar:
three roundings of 2^-24 on values whose layer sums stay within a factor
sqrt(size) of their terms -- 1e-5 of the largest score), and the choice is
their argmin."""

import numpy as np
import pytest
import torch

from tests._util import to_dev

pytestmark = pytest.mark.gpu

from flagsparse_public_amd import _lib  # noqa: E402
from flagsparse_public_amd.selector import Mlp  # noqa: E402

DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("in_dim,hidden,out", [(16, 64, 18), (1, 1, 1), (16, 96, 11), (16, 101, 3),
                                               (16, 102, 18), (40, 256, 256)])
def test_scores_and_choice(orc, in_dim, hidden, out):
    rng = np.random.default_rng(hidden)
    mlp = Mlp(out, DEV, hidden=hidden, in_dim=in_dim, seed=3)
    mu = rng.normal(size=in_dim).astype(np.float32)
    sd = rng.uniform(0.5, 2, in_dim).astype(np.float32)
    choice = torch.empty(1, dtype=torch.int32, device=DEV)
    scores = torch.empty(out, dtype=torch.float32, device=DEV)
    for _ in range(3):
        x = rng.normal(size=in_dim).astype(np.float32)
        _lib.mlp_select(mlp.net, to_dev(x), to_dev(mu), to_dev(sd), choice, scores, DEV)
        want = orc.mlp_forward(((x - mu) / sd)[None].astype(np.float64), *mlp.unpack())[2][0]
        got = scores.cpu().numpy()
        assert np.max(np.abs(got - want)) <= 1e-5 * max(1.0, np.max(np.abs(want)))
        assert choice.item() == int(np.argmin(got))
