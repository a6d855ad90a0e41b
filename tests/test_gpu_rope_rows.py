"""The 16-byte form of qk_rope_cache against the general one (a wave per head) on the same inputs.

The general form runs when a pointer is not 16-byte aligned, so each case runs twice, the second time
on a copy of the packed rows that starts 4 bytes into its allocation. Only the order of the 32-bit sum
of squares differs, which moves inv_std by an ulp of FP32 and with it, rarely, a rounding; values and
untouched slots agree bit for bit.
"""

import pytest
import torch

from conftest import to_bits
from kernels import qk_rope as R

pytestmark = pytest.mark.gpu


class Norm:
    def __init__(self, weight, eps):
        self.weight, self.variance_epsilon = weight, eps


def _inputs(b, t, hq, hkv, d, cap, device, seed=0):
    g = torch.Generator(device=device).manual_seed(seed)

    def rnd(*shape, scale=1.0, shift=0.0):
        return (torch.randn(*shape, generator=g, device=device) * scale + shift).to(torch.bfloat16)

    packed = rnd(b, t, (hq + 2 * hkv) * d, scale=2.0)
    norms = Norm(rnd(d, scale=0.1, shift=1.0), 1e-6), Norm(rnd(d, scale=0.1, shift=1.0), 2e-6)
    return packed, norms, rnd(b, hkv, cap, d), rnd(b, hkv, cap, d)


def _offset_copy(x):
    """The same values, 4 bytes past a 16-byte boundary."""
    flat = torch.empty(x.numel() + 2, dtype=x.dtype, device=x.device)
    out = flat[2:].view(x.shape)
    out.copy_(x)
    assert out.data_ptr() % 16 == 4
    return out


def _table(rows, d, device):
    angle = torch.rand(rows, d // 2, device=device, generator=torch.Generator(device=device).manual_seed(9)) * 6.28
    angle = torch.cat((angle, angle), dim=-1)
    return angle.cos().to(torch.bfloat16), angle.sin().to(torch.bfloat16)


def _both(packed, norms, keys, values, run):
    got = []
    for rows in (packed, _offset_copy(packed)):
        k, v = keys.clone(), values.clone()
        got.append((run(rows, norms, k, v), k, v))
    (q, k, v), (wq, wk, wv) = got
    # n = bf16(x inv_std) may be one BF16 ulp apart (2^-7), w = bf16(n gain) and its product with cos or sin round
    # twice more each (2^-9 every time): 2^-6 of |w cos| + |w' sin|, which is at most the norm of the pair that is
    # rotated (cos^2 + sin^2 = 1, to the table's own rounding); the sum's two roundings add 2^-8 of that.
    for a, w in ((q, wq), (k, wk)):
        a, w = a.float(), w.float()
        half = w.shape[-1] // 2
        pair = torch.hypot(w[..., :half], w[..., half:])
        pair = torch.cat((pair, pair), dim=-1)
        assert bool(((a - w).abs() <= 1.02 * (2.0 ** -6 + 2.0 ** -8) * pair).all())
        assert float((a != w).float().mean()) < 2e-3  # inv_std moves by an ulp of FP32: few results round apart
    assert (to_bits(v) == to_bits(wv)).all()
    return got[0]


# heads that fill a workgroup's groups exactly, by one more and one less, few enough for several rows a
# workgroup (the last one ragged), and beyond four passes; rows below and above the 1024-workgroup line.
@pytest.mark.parametrize("b,t,hq,hkv,d", [(1, 1, 1, 1, 128), (3, 1, 4, 1, 128), (1, 5, 14, 1, 128), (1, 3, 15, 1, 128),
                                          (2, 700, 32, 8, 128), (1, 4097, 4, 1, 128), (1, 1030, 13, 2, 128),
                                          (1, 1025, 80, 8, 128), (5, 3, 2, 1, 64), (1, 1029, 40, 8, 64),
                                          (1, 1, 64, 8, 64), (3, 1500, 2, 2, 64)])
def test_prefill_matches_the_general_form(cuda, b, t, hq, hkv, d):
    packed, norms, keys, values = _inputs(b, t, hq, hkv, d, t + 3, cuda)
    cos, sin = (x[None] for x in _table(t, d, cuda))
    position = torch.arange(t, device=cuda, dtype=torch.int64)
    _, k, v = _both(packed, norms, keys, values,
                    lambda x, n, kc, vc: R.qk_rope_cache(x, *n, cos, sin, position, kc, vc, hq, prefill=True))
    assert (to_bits(k[:, :, t:]) == to_bits(keys[:, :, t:])).all()
    heads = packed.view(b, t, -1, d)[:, :, hq + hkv:].transpose(1, 2)
    assert (to_bits(v[:, :, :t]) == to_bits(heads)).all()


@pytest.mark.parametrize("d,hq,hkv", [(128, 16, 8), (64, 3, 1)])
def test_steps_at_their_own_positions_and_limits(cuda, d, hq, hkv):
    b, t, cap, rows = 4, 2, 24, 40
    packed, norms, keys, values = _inputs(b, t, hq, hkv, d, cap, cuda, seed=1)
    cos, sin = _table(rows, d, cuda)
    # A row inside, one whose second slot is past the cache, one past it, one before it (phase inside).
    position = torch.tensor([3, cap - 1, cap + 4, -2], device=cuda)
    phases = torch.tensor([[0, 1], [0, 1], [0, 1], [5, 6]], device=cuda)
    q, k, v = _both(packed, norms, keys, values,
                    lambda x, n, kc, vc: R.qk_rope_cache(x, *n, cos, sin, position, kc, vc, hq, rows=True,
                                                         phases=phases))
    for new, old in ((k, keys), (v, values)):
        kept = torch.ones((b, cap), dtype=torch.bool, device=cuda)
        kept[0, 3:5], kept[1, cap - 1] = False, False
        assert (to_bits(new.transpose(1, 2)[kept]) == to_bits(old.transpose(1, 2)[kept])).all()
        assert not torch.equal(new[0, :, 3:5], old[0, :, 3:5])
    # A phase outside the table leaves the row's slots alone.
    phases = torch.full((b, t), rows, device=cuda, dtype=torch.int64)
    k2, v2 = keys.clone(), values.clone()
    R.qk_rope_cache(packed, *norms, cos, sin, torch.zeros_like(position), k2, v2, hq, rows=True, phases=phases)
    assert (to_bits(k2) == to_bits(keys)).all() and (to_bits(v2) == to_bits(values)).all()
