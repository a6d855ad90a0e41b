"""qk_rope_cache on both sides of the line below which few heads of 64 take the general form: there the
aligned rows give the same bits as the same rows 4 bytes further, above it they agree as the two forms do."""

import pytest
import torch

from conftest import to_bits
from test_gpu_rope_rows import _both, _inputs, _offset_copy, _table

from kernels import qk_rope as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,hq,hkv,few", [(1, 1, 1, True), (127, 14, 3, True), (128, 14, 3, False), (32, 64, 8, False),
                                             (31, 64, 8, True)])
def test_few_heads_of_64(cuda, rows, hq, hkv, few):
    packed, norms, keys, values = _inputs(rows, 1, hq, hkv, 64, 9, cuda, seed=rows)
    cos, sin = _table(16, 64, cuda)
    position = torch.arange(rows, device=cuda) % 9
    phases = torch.full((rows, 1), 3, dtype=torch.int64, device=cuda)
    run = lambda x, n, k, v: R.qk_rope_cache(x, *n, cos, sin, position, k, v, hq, rows=True, phases=phases)
    if not few:
        _both(packed, norms, keys, values, run)
        return
    got = [keys.clone(), values.clone()]
    want = [keys.clone(), values.clone()]
    got.append(run(packed, norms, *got))
    want.append(run(_offset_copy(packed), norms, *want))
    for a, b in zip(got, want):
        assert (to_bits(a) == to_bits(b)).all()
