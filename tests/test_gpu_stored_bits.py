"""Stored BF16 bits: nearest-even over special and random FP32 values, every NaN as 0x7FC0."""

import numpy as np
import pytest
import torch

from conftest import to_bits
from kernels import rmsnorm as N
from kernels.merged import Split, materialize
from kernels.swiglu import swiglu

pytestmark = pytest.mark.gpu


def _words(n):
    """Every sign and exponent with mantissas at and around the rounding ties, then random words."""
    low = np.array([0, 1, 0x7FFF, 0x8000, 0x8001, 0xFFFF, 0x17FFF, 0x18000, 0x18001, 0x7FFFFF], dtype=np.uint32)
    high = np.arange(512, dtype=np.uint32) << 23
    words = (high[:, None] | low[None, :]).reshape(-1)
    rest = np.random.default_rng(0).integers(0, 2 ** 32, n - words.size, dtype=np.uint64).astype(np.uint32)
    return np.concatenate((words, rest))


def _want(words):
    """Round to nearest even in integers; NaN as 0x7FC0."""
    w = words.astype(np.uint64)
    out = ((w + 0x7FFF + ((w >> 16) & 1)) >> 16).astype(np.uint16)
    return np.where((words & 0x7FFFFFFF) > 0x7F800000, np.uint16(0x7FC0), out)


def test_one_value_stores(cuda):
    words = _words(8192)
    x = torch.from_numpy(words.view(np.float32).copy()).to(cuda).view(1, 1, -1)
    np.testing.assert_array_equal(to_bits(materialize(Split(x, (1, x.shape[-1])))).reshape(-1), _want(words))


@pytest.mark.parametrize("splits", [2, 3])
def test_pair_stores(cuda, splits):
    """add_rms_norm's sum over FP32 partial planes (the further ones zero) and a zero residual."""
    words = _words(8192)
    x = torch.zeros((splits, 1, 8192), device=cuda)
    x[0, 0] = torch.from_numpy(words.view(np.float32).copy())
    zero = torch.zeros((1, 8192), dtype=torch.bfloat16, device=cuda)
    _, total = N.add_rms_norm(Split(x, (1, 8192)), zero, torch.ones(8192, dtype=torch.bfloat16, device=cuda), 1e-6)
    want = _want(words)
    np.testing.assert_array_equal(to_bits(total).reshape(-1), np.where(want == 0x8000, np.uint16(0), want))


# widths whose group count per row is one, a power of two, and neither; rows so the last block is ragged.
@pytest.mark.parametrize("rows,width", [(1, 8), (3, 8), (257, 24), (31, 2048), (7, 12296), (1000, 1544)])
def test_swiglu_rows_and_their_specials(cuda, rows, width):
    g = torch.Generator(device=cuda).manual_seed(rows + width)
    packed = (torch.randn((rows, 2 * width), generator=g, device=cuda) * 4).to(torch.bfloat16)
    packed[0, :4] = torch.tensor([float("inf"), -float("inf"), float("nan"), -200.0])
    packed[-1, width:width + 2] = torch.tensor([float("nan"), float("inf")])
    got = swiglu(packed)
    gate, up = packed.float().chunk(2, dim=-1)
    want = ((gate / (1 + torch.exp(-gate))).to(torch.bfloat16).float() * up).to(torch.bfloat16)
    nan = want.isnan()
    assert (to_bits(got)[nan.cpu().numpy()] == 0x7FC0).all()
    a, w = got[~nan].float(), want[~nan].float()
    # exp and the division may differ by FP32 ulps: SiLU, and then the product, one BF16 ulp each way.
    close = (a == w) | ((a - w).abs() <= 2.0 ** -6 * w.abs())
    assert bool(close.all()) and float((a != w).float().mean()) < 1e-3
