"""GPU parity of the decode attention's tile kernel (ftk_attn_tile.hip) at the edges of its units and intervals.

A unit is 32 cache slots; the interval of a split is the row's own share of
min(position + 1, capacity), in whole units; up to 32 slots per wave of the
full cache, D = 128 and up to 4 heads per KV head stay with the QUAD kernel.
Rows of one batch stand at different places, NaN in every slot they can't see.
Against the oracle, as tests/test_gpu_attention.py: |y - ref| <= 2e-2 +
1e-2 |ref| (values ~ N(0, 1): p rounded to BF16, 2^-9 relative, plus the
output's own rounding stay well inside it).
"""

import pytest
import torch

from conftest import to_bits
from test_gpu_attention import _inputs, _oracle, cfg, within
from test_gpu_rope_attention import D, _case, _check_caches, _fused
from test_gpu_rope_attention import _oracle as _rope_oracle

from kernels import decode_attention as A

pytestmark = pytest.mark.gpu

POSITIONS = [0, 30, 31, 32, 127, 128, 191, 400]  # 400: past the cache, every slot visible


@pytest.mark.parametrize("splits,waves", [(1, 4), (1, 8), (2, 4), (3, 4), (7, 8)])
@pytest.mark.parametrize("dim,groups", [(128, 1), (128, 3), (128, 4), (128, 5), (128, 8), (64, 1), (64, 4), (64, 7)])
def test_ragged_rows(cuda, dim, groups, splits, waves):
    b, hkv, cap, scale = len(POSITIONS), 2, 300, dim ** -0.5
    q, k, v = _inputs(b, hkv, dim, cap, groups, 1.0, 7 * groups + splits, cuda)
    for i, p in enumerate(POSITIONS):
        k[i, :, p + 1:] = float("nan")
        v[i, :, p + 1:] = float("nan")
    position = torch.tensor(POSITIONS, device=cuda)
    got = to_bits(A.attend(q.reshape(b, hkv * groups, dim), k, v, position, scale, cfg(splits=splits, waves=waves)))
    for i, p in enumerate(POSITIONS):
        want = _oracle(q[i:i + 1], k[i:i + 1], v[i:i + 1], min(p, cap - 1), scale)
        assert within(got.reshape(b, hkv * groups, dim)[i:i + 1], want), f"row {i}, position {p}"


@pytest.mark.parametrize("cap,splits,waves", [(128, 1, 4), (129, 1, 4), (256, 1, 8), (257, 1, 8), (300, 2, 4)])
@pytest.mark.parametrize("groups", [1, 4])
def test_head_norm_and_rotation(cuda, cap, splits, waves, groups):
    """Both sides of the line between QUAD and the tile kernel, the new slot in each wave's and each split's place."""
    positions, hkv, scale = [0, 31, 32, cap // 2, cap - 1, cap], 2, D ** -0.5
    c = _case(len(positions), hkv * groups, hkv, cap, positions, seed=cap + groups, device=cuda)
    before_k, before_v = to_bits(c["keys"]), to_bits(c["values"])
    want, want_k, want_v = _rope_oracle(c, hkv * groups, scale)
    got = to_bits(_fused(c, hkv * groups, scale, cfg(splits=splits, waves=waves)))
    assert within(got.reshape(want.shape), want)
    _check_caches(c, before_k, before_v, want_k, want_v)
