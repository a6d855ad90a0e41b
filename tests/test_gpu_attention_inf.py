"""Infinite cached values in slots a row sees: the output's dimension is that infinity, as the product
of the softmax's weight with it is, and every other dimension keeps its bits.

The largest score of each head (p = 1), the newest slot and slots with smaller weights, on both sides
of the line between the QUAD and the tile kernel, with one and several intervals, at both dimensions.
Scores ~ N(0, 1), so every weight is far from underflow.
"""

import pytest
import torch

from conftest import to_bits
from test_gpu_attention import _inputs, cfg
from test_gpu_rope_attention import D, _case, _fused

from kernels import decode_attention as A

pytestmark = pytest.mark.gpu


def _spread(slots, dim):
    """(slot, dimension, infinity) with a dimension of its own for each slot, every second dimension used."""
    return [(slot, 2 * i, float("inf") if i % 3 else float("-inf")) for i, slot in enumerate(slots[:dim // 2])]


def _expect(got, base, marks):
    dims = [d for _, d, _ in marks]
    for _, d, inf in marks:
        assert bool((got[..., d] == inf).all()), f"dimension {d}: {got[..., d].flatten()[:4].tolist()}, not {inf}"
    rest = [d for d in range(got.shape[-1]) if d not in dims]
    assert (to_bits(got[..., rest].contiguous()) == to_bits(base[..., rest].contiguous())).all()


@pytest.mark.parametrize("cap,splits,waves", [(128, 1, 4), (129, 1, 4), (300, 1, 8), (300, 3, 4)])
@pytest.mark.parametrize("dim,groups", [(128, 1), (128, 4), (128, 8), (64, 4)])
def test_infinite_values_stay_infinite(cuda, dim, groups, cap, splits, waves):
    q, k, v = _inputs(1, 1, dim, cap, groups, 1.0, 31 * groups + cap, cuda)
    top = (q.float().view(groups, dim) @ k[0, 0].float().t()).argmax(dim=-1).tolist()
    slots = list(dict.fromkeys(top + [cap - 1, 0] + list(range(5, cap, 13))))
    marks = _spread(slots, dim)
    position = torch.tensor([cap - 1], device=cuda)
    run = lambda values: A.attend(q.reshape(1, groups, dim), k, values, position, dim ** -0.5,
                                  cfg(splits=splits, waves=waves))
    inf = v.clone()
    for slot, d, value in marks:
        inf[0, 0, slot, d] = value
    _expect(run(inf), run(v), marks)


@pytest.mark.parametrize("cap", [100, 300])
def test_infinite_values_beside_the_new_slot(cuda, cap):
    """The fused prologue: cached infinities, and one in the step's own value head."""
    hq, hkv = 4, 1
    c = _case(1, hq, hkv, cap, [cap - 1], seed=cap, device=cuda)
    marks = _spread(list(range(0, cap - 1, 7)), D - 2)
    inf = {name: t.clone() for name, t in c.items()}
    for slot, d, value in marks:
        inf["values"][0, 0, slot, d] = value
    inf["packed"][0, (hq + hkv) * D + D - 2] = float("-inf")
    run = lambda x: _fused(x, hq, D ** -0.5, cfg(splits=1, waves=4))
    _expect(run(inf), run(c), marks + [(cap - 1, D - 2, float("-inf"))])
