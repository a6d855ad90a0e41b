"""GPU parity of the FLOW kind and the MFMA kind's LDS-fed form, by explicit launch choice and by default.

Sizes stand where these kernels change: x row counts at the edges of their builds (4, 8, 16, 24, 32),
K below one segment, ragged in the last segment, with a wave short of a segment and at FLOW's largest,
N below, at and past a tile. Tolerance: |y - ref| <= 2e-2 + 1e-2|ref| against the oracle, as the other
kinds (FP32 sums, BF16 results of size ~1 at these scales)."""

import numpy as np
import pytest
import torch

from conftest import seeded, to_bits
from oracle import bf16, path

from kernels import _native
from kernels import argmax as A
from kernels import linear as L
from kernels import swiglu as S

pytestmark = pytest.mark.gpu

EPS = 1e-6
FLOW = _native.Config(_native.KIND_FLOW, 16, 0, 0, 0)
TILES = ((8, 8), (12, 8), (16, 8), (20, 8), (24, 8), (16, 4), (24, 4), (32, 4))


def tile(rows, waves):
    return _native.Config(_native.KIND_MFMA, rows, 1, 0, waves)


def within(got, want_bits):
    g, w = bf16.to_f32(to_bits(got)).astype(np.float64), bf16.to_f32(want_bits).astype(np.float64)
    return bool(np.all(np.abs(g - w) <= 2e-2 + 1e-2 * np.abs(w)))


def inputs(m, n, k, device, seed):
    return (seeded((m, k), seed=seed, device=device), seeded((n, k), seed=seed + 1, scale=0.02, device=device),
            seeded((k,), seed=seed + 2, scale=0.1, shift=1.0, device=device))


#: (M, N, K)
SHAPES = [(1, 33, 8), (4, 5000, 1000), (5, 16, 128), (8, 4112, 1032), (9, 600, 2560), (16, 300, 5120), (17, 48, 136),
          (24, 5000, 1160), (25, 1000, 5120), (32, 4100, 3968)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("norm", [False, True])
def test_flow_matches_oracle(cuda, m, n, k, norm):
    x, w, g = inputs(m, n, k, cuda, 9000 + m)
    xb, wb, gb = to_bits(x), to_bits(w), to_bits(g)
    gain = g if norm else None
    y = L.rms_norm_linear(x, g, EPS, w, config=FLOW) if norm else L.project(x, w, FLOW)
    assert within(y, path.norm_project(xb, gb, EPS, wb) if norm else path.project(xb, wb))
    ids, logits = A.lm_head_argmax(x, w, gain, EPS, config=FLOW)
    assert torch.equal(logits, y)
    np.testing.assert_array_equal(ids.cpu().numpy(), path.argmax_first(to_bits(logits)))
    pairs = w if n % 2 == 0 else w[:-1].contiguous()
    act = S.gate_up_swiglu(x, pairs, gain, EPS, config=FLOW)
    assert within(act, path.gate_up_swiglu(xb, to_bits(pairs), gb if norm else None, EPS))


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("rows,waves", TILES)
def test_tiles_match_oracle(cuda, m, n, k, rows, waves):
    x, w, g = inputs(m, n, k, cuda, 9100 + m)
    cfg = tile(rows, waves)
    if m > 24 and (rows, waves) == (24, 8):  # 32 x rows beside 24 weight rows: four waves only
        with pytest.raises(_native.FtkError):
            L.project(x, w, cfg)
        return
    y = L.project(x, w, cfg)
    assert within(y, path.project(to_bits(x), to_bits(w)))
    r = seeded((m, n), seed=9200 + m, device=cuda)
    assert torch.equal(L.linear_residual(x, w, r, config=cfg), (y.float() + r.float()).to(torch.bfloat16))
    assert within(L.rms_norm_linear(x, g, EPS, w, config=cfg), path.norm_project(to_bits(x), to_bits(g), EPS, to_bits(w)))
    if rows == 32 and n % 2 == 0:
        assert within(S.gate_up_swiglu(x, w, g, EPS, config=cfg), path.gate_up_swiglu(to_bits(x), to_bits(w), to_bits(g), EPS))
    if rows in (16, 32):
        ids, logits = A.lm_head_argmax(x, w, None, EPS, config=cfg)
        assert torch.equal(logits, y)
        np.testing.assert_array_equal(ids.cpu().numpy(), path.argmax_first(to_bits(logits)))


@pytest.mark.parametrize("cfg", [FLOW, tile(8, 8), tile(20, 8), tile(32, 4)])
def test_infinities_and_nan_stay_in_their_row_and_column(cuda, cfg):
    """A ragged K reads past a row's end into the next row, and operands of rows that do not exist read
    other data: neither may reach a result. An infinite weight gives infinite outputs, as summed."""
    m, n, k = 5, 70, 136
    x, w, _ = inputs(m, n, k, cuda, 9300)
    x = x.abs() + 0.1
    want = L.project(x, w, cfg)
    w2, x2 = w.clone(), x.clone()
    w2[7], w2[n - 1] = float("nan"), float("nan")
    w2[20, k - 1] = float("inf")
    x2[2] = float("nan")
    got = L.project(x2, w2, cfg)
    assert bool(got[2].isnan().all()) and bool(got[:, 7].isnan().all()) and bool(got[:, n - 1].isnan().all())
    rows, cols = [0, 1, 3, 4], [c for c in range(n) if c not in (7, 20, n - 1)]
    assert bool((got[rows, 20] == float("inf")).all())
    assert torch.equal(got[rows][:, cols], want[rows][:, cols])


@pytest.mark.parametrize("m", [2, 4, 5, 16, 17, 32])
def test_defaults_match_oracle(cuda, m):
    """The default launches where these kernels are chosen (K = 1920, a wide and a narrow projection)."""
    h, q, i = 1920, 4096, 2048
    x, w, g = inputs(m, q, h, cuda, 9400 + m)
    assert within(L.rms_norm_linear(x, g, EPS, w), path.norm_project(to_bits(x), to_bits(g), EPS, to_bits(w)))
    assert within(L.linear(x, w), path.project(to_bits(x), to_bits(w)))
    assert within(S.gate_up_swiglu(x, w, g, EPS), path.gate_up_swiglu(to_bits(x), to_bits(w), to_bits(g), EPS))
    ids, logits = A.lm_head_argmax(x, w, g, EPS)
    assert within(logits, path.norm_project(to_bits(x), to_bits(g), EPS, to_bits(w)))
    np.testing.assert_array_equal(ids.cpu().numpy(), path.argmax_first(to_bits(logits)))
    act = seeded((m, i), seed=9500 + m, device=cuda)
    down = seeded((h, i), seed=9501, scale=0.02, device=cuda)
    r = seeded((m, h), seed=9502, device=cuda)
    want = bf16.round_bits(bf16.to_f32(path.project(to_bits(act), to_bits(down))) + bf16.to_f32(to_bits(r)))
    assert within(L.linear_residual(act, down, r), want)


def test_embedding_rows_through_flow(cuda):
    """The gather prologue: the stored rows are the table's, ids past it clamped."""
    table, w, g = inputs(300, 512, 1920, cuda, 9600)
    ids = torch.tensor([299, 0, 300, -1, 7, 7], dtype=torch.int64, device=cuda)
    y, hidden = L.embed_rms_norm_linear(ids, table, g, EPS, w, config=FLOW)
    rows = table[ids.clamp(0, 299)]
    assert torch.equal(hidden, rows)
    assert torch.equal(y, L.rms_norm_linear(rows, g, EPS, w, config=FLOW))
