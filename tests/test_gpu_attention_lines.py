"""Decode attention on both sides of the lines between the QUAD and the tile kernel that go by rows and
heads per KV head: one row over long intervals, several rows over two units per wave. Against the oracle,
NaN in every slot from the position on, as tests/test_gpu_rope_attention.py."""

import pytest

from conftest import to_bits
from test_gpu_attention import cfg, within
from test_gpu_rope_attention import D, _case, _check_caches, _fused
from test_gpu_rope_attention import _oracle as _rope_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap,splits,waves", [(512, 2, 4), (514, 2, 4), (700, 2, 4), (1300, 2, 8), (257, 1, 4)])
@pytest.mark.parametrize("groups", [1, 2, 4])
@pytest.mark.parametrize("where", [[0], [255], [256], [-1], [0, 256, -1]])
def test_lines_by_rows_and_heads(cuda, where, groups, cap, splits, waves):
    hkv, scale = 2, D ** -0.5
    positions = [p if p >= 0 else cap + p for p in where]
    c = _case(len(positions), hkv * groups, hkv, cap, positions, seed=cap + groups, device=cuda)
    before_k, before_v = to_bits(c["keys"]), to_bits(c["values"])
    want, want_k, want_v = _rope_oracle(c, hkv * groups, scale)
    got = to_bits(_fused(c, hkv * groups, scale, cfg(splits=splits, waves=waves)))
    assert within(got.reshape(want.shape), want)
    _check_caches(c, before_k, before_v, want_k, want_v)
