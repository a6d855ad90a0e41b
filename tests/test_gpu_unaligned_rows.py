"""linear() from 17 rows on rows or weights that are not 16-byte aligned: torch's own result, bit for bit."""

import pytest
import torch
from torch.nn import functional as F

from conftest import seeded

from kernels import linear as L

pytestmark = pytest.mark.gpu


def _shifted(t):
    """The same values, two bytes past a 16-byte boundary."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    out = flat[1:].view(t.shape)
    out.copy_(t)
    assert out.data_ptr() % 16 == 2
    return out


@pytest.mark.parametrize("m", [17, 24, 32])
@pytest.mark.parametrize("shift_x,shift_w", [(True, False), (False, True), (True, True)])
def test_unaligned_operands(cuda, monkeypatch, m, shift_x, shift_w):
    monkeypatch.setattr(L, "TUNE", False)
    monkeypatch.setattr(L, "_CHOICES", {})
    x, w = seeded((m, 2048), seed=m, device=cuda), seeded((1536, 2048), seed=1, scale=0.02, device=cuda)
    assert L.default_choice("linear", m, 1536, 2048) is None  # aligned, this library's kernels
    x, w = _shifted(x) if shift_x else x, _shifted(w) if shift_w else w
    assert torch.equal(L.linear(x, w), F.linear(x, w))
    assert torch.equal(L.linear(x[None], w), F.linear(x[None], w))
