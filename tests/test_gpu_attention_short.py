"""Short caches, attended in one launch: around the lines of the planner's rule, against 64 bits."""

import pytest
import torch

from kernels import decode_attention as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (8, 8, 128), (16, 2, 128), (8, 2, 64)])
@pytest.mark.parametrize("b,capacity,one", [(1, 129, True), (1, 256, True), (2, 65, True), (3, 256, True), (3, 257, None),
                                            (3, 384, None), (64, 384, True), (64, 385, None)])
def test_short_caches(cuda, hq, hkv, d, b, capacity, one):
    p = A.plan(b, hq, hkv, capacity, d)
    if one is not None:
        assert p.splits == 1 and p.workspace_bytes == 0
    g = torch.Generator(device=cuda).manual_seed(capacity + hq)
    q, k, v = (torch.randn(shape, generator=g, device=cuda).to(torch.bfloat16)
               for shape in ((b, hq, d), (b, hkv, capacity, d), (b, hkv, capacity, d)))
    # Rows at the start, the end and past the end of their caches, the rest spread between.
    position = torch.linspace(0, capacity - 1, b, device=cuda).long()
    if b > 2:
        position[1] = capacity + 3
    for row, last in enumerate(position.tolist()):
        k[row, :, last + 1:] = float("nan")
        v[row, :, last + 1:] = float("nan")
    out = A.attend(q, k, v, position, d ** -0.5).view(b, hq, d)
    for row, last in enumerate(position.tolist()):
        n = min(last + 1, capacity)
        query = q[row].double().view(hkv, -1, d)
        prob = ((query @ k[row, :, :n].double().transpose(1, 2).contiguous()) * d ** -0.5).softmax(dim=-1)
        values = v[row, :, :n].double()
        want, size = (prob @ values).view(hq, d), (prob @ values.abs()).view(hq, d)
        # The output rounds once and p once (half an ulp, 2^-9 each), the 32-bit sums stay far below.
        bound = 2.0 ** -9 * want.abs() + 2.0 ** -9 * size + 2.0 ** -14 * size
        assert bool(((out[row].double() - want).abs() <= bound).all())
