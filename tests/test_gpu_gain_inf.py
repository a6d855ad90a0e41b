"""An infinite gain in the last elements of a ragged K: each row's outputs are the infinity that its x and
the weights make of it, in FLOW as in the LDS-fed form. What the kernels read past K must not turn it into
NaN (FLOW's gain there is the last elements again)."""

import pytest
import torch

from conftest import seeded

from kernels import _native
from kernels import linear as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg", [_native.Config(_native.KIND_FLOW, 16, 0, 0, 0), _native.Config(_native.KIND_MFMA, 16, 1, 0, 8)])
@pytest.mark.parametrize("m,k", [(1, 136), (5, 136), (8, 1032), (17, 1160), (32, 4104)])
@pytest.mark.parametrize("back", [1, 8])
def test_infinite_gain_at_a_ragged_end(cuda, cfg, m, k, back):
    n = 70
    x = seeded((m, k), seed=m, device=cuda)
    w = seeded((n, k), seed=k, scale=0.02, device=cuda)
    g = seeded((k,), seed=7, scale=0.1, shift=1.0, device=cuda)
    x = torch.where(x == 0, torch.ones_like(x), x)
    w = torch.where(w == 0, torch.ones_like(w), w)
    g[k - back] = float("inf")
    got = L.rms_norm_linear(x, g, 1e-6, w, config=cfg)
    sign = x[:, k - back].float().sign()[:, None] * w[:, k - back].float().sign()[None, :]
    assert torch.equal(got.float(), sign * float("inf"))
