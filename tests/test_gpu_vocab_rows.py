"""lm_head + argmax from 17 rows: the FLOW walk, without a norm too, and the norm in a launch of its own
past K = 4096. Logits within 2e-2 + 1e-2 |ref| of FP32 (FP32 sums, BF16 results of size ~1), ids the first
maximum of them."""

import numpy as np
import pytest
import torch

from conftest import seeded, to_bits
from oracle import path

from kernels import _native
from kernels import argmax as A
from kernels import linear as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [17, 24, 32])
@pytest.mark.parametrize("v,k,norm,apart", [(9001, 512, False, False), (4100, 1024, True, False), (3000, 4096, True, False),
                                            (2056, 4104, True, True), (2056, 5120, True, True), (2056, 5120, False, False)])
def test_vocabulary_from_17_rows(cuda, monkeypatch, m, v, k, norm, apart):
    x = seeded((m, k), seed=m, device=cuda)
    w = seeded((v, k), seed=k, scale=0.02, device=cuda)
    g = seeded((k,), seed=3, scale=0.1, shift=1.0, device=cuda) if norm else None
    monkeypatch.setattr(L, "TUNE", False)
    calls, launch = [], L.fused_project

    def spy(*args, **kwargs):
        calls.append((kwargs["config"].kind if kwargs["config"] is not None else None, args[4] is not None))
        return launch(*args, **kwargs)

    monkeypatch.setattr(L, "fused_project", spy)
    top = torch.empty(m, dtype=torch.float32, device=cuda)
    ids, logits = A.lm_head_argmax(x, w, g, 1e-6, top=top)
    assert calls == [(_native.KIND_FLOW, norm and not apart)]
    rows = x.float()
    if norm:
        rows = (rows * torch.rsqrt(rows.square().mean(-1, keepdim=True) + 1e-6)).to(torch.bfloat16)
        rows = (rows * g).float()
    want = rows @ w.float().t()
    assert bool(((logits.float() - want).abs() <= 2e-2 + 1e-2 * want.abs()).all())
    np.testing.assert_array_equal(ids.cpu().numpy(), path.argmax_first(to_bits(logits)))
    assert torch.equal(top, logits.float().gather(1, ids[:, None])[:, 0])
