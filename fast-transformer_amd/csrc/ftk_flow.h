// M = 1..32 skinny BF16 projection, FLOW kind: a persistent walk over 16-row weight tiles for any
// K % 8 == 0 to 5120, the x rows in registers throughout (device code; ftk_flow_x*.hip instantiate it).
//
// Same sums, roundings and fused extras as the other kinds (engine/kernels/linear.py:50-78
// _skinny_gemm; RMSNorm prologue engine/kernels/rmsnorm.py:21-46; SwiGLU
// engine/kernels/swiglu.py:13-24; greedy argmax engine/kernels/argmax.py:19-48).
//
// What bounds it: HBM for the weights, and before the first product a chain every workgroup runs:
// x from L2 (all workgroups read the same rows at once, ~2 us), their sums and a barrier (~1 us),
// the normalisation on the VALU (K = 4096: 1.4 us to 16 x rows, 3.8 us to 32; its ten operations per
// pair of values have no packed form here). Measured with those parts left out.
//
// Layout and schedule:
//   * The 128-wide K segments are dealt to 8 waves (wave kw: kw, kw + 8, ...), so any K divides; the
//     last segment may be short (its operands are zeroed past K) and the last wave may have one fewer.
//   * x is loaded once, 4 rows x 256 bytes per wave instruction straight into LDS (the RING kind's
//     swizzled layout), read as MFMA B operands and kept: 16 registers per segment and 16 rows (two
//     column blocks past 16 rows). The norm's sums are taken from those operands, which are then
//     normalised in place, so x is neither read twice nor normalised per tile.
//   * The same LDS is then the weight ring: four units (16 rows x 256 bytes) in flight per wave,
//     waited for with exact vmcnts, refilled as soon as they are in registers; no barrier but the one
//     before an epilogue. Units whose slots lie past the staged x are in flight from the start.
//     (The units under the staged x loaded into registers meanwhile: slower, 17.3 -> 18.5 us at
//     6144 x 4096 and 24 rows; the weights' burst delays x. Tiles of 8 and 12 rows: slower too.)
//   * Tiles and epilogues as RING's: partials parked in LDS and summed in wave order.
//
// us per graph node on MI355X over distinct weights, with the norm, against the launches these shapes
// had: gate/up 19456 x 2560 at 8 / 16 / 24 rows 20.0 / 19.5 / 23.7 against 29.9 / 34.7 / 30.2 (5.1 TB/s
// at 16 rows), 6144 x 1024 5.8 / 6.3 / 8.2 against
// 7.5 / 8.5 / 16.7, lm_head 151936 x 1024 54.8 / 54.9 / 71 against 184 / 228 / 81. At K = 4096 and up
// to 16 rows the RING kind, built for that K, stays ahead (6144 x 4096 11.2 / 12.6 against 12.5 / 13.1).
#pragma once

#include <type_traits>

#include "ftk_dma.h"
#include "ftk_internal.h"

namespace ftk {

// The MFMA operand chunks s = 0..3 of 16 rows in LDS, read and waited for in one block.
__device__ __forceinline__ void read_rows16(const uint32_t (&at)[4], u32x4_t (&v)[4]) {
  asm volatile(
      "ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %6\n\tds_read_b128 %3, %7\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
      : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3])
      : "memory");
}
__device__ __forceinline__ void read_gain4(uint32_t at, u32x4_t (&g)[4]) {
  asm volatile(
      "ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:64\n\tds_read_b128 %2, %4 offset:128\n\t"
      "ds_read_b128 %3, %4 offset:192\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(g[0]), "=&v"(g[1]), "=&v"(g[2]), "=&v"(g[3])
      : "v"(at)
      : "memory");
}
__device__ __forceinline__ void ds_put(uint32_t at, float v) {
  asm volatile("ds_write_b32 %0, %1" ::"v"(at), "v"(v) : "memory");
}
// Sum of eight floats in LDS, STRIDE bytes apart, in order.
template <int STRIDE>
__device__ __forceinline__ float ds_sum8(uint32_t at) {
  float v[8];
  asm volatile(
      "ds_read_b32 %0, %8\n\tds_read_b32 %1, %8 offset:%9\n\tds_read_b32 %2, %8 offset:%10\n\t"
      "ds_read_b32 %3, %8 offset:%11\n\tds_read_b32 %4, %8 offset:%12\n\tds_read_b32 %5, %8 offset:%13\n\t"
      "ds_read_b32 %6, %8 offset:%14\n\tds_read_b32 %7, %8 offset:%15\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
      : "v"(at), "n"(STRIDE), "n"(2 * STRIDE), "n"(3 * STRIDE), "n"(4 * STRIDE), "n"(5 * STRIDE), "n"(6 * STRIDE),
        "n"(7 * STRIDE)
      : "memory");
  float total = v[0];
#pragma unroll
  for (int i = 1; i < 8; ++i) total += v[i];
  return total;
}

// Wait until at most min(units, A) units of WL loads are outstanding.
template <int A, int WL>
__device__ __forceinline__ void wait_units(int units) {
  if constexpr (A == 0) {
    wait_vm<0>();
  } else {
    if (units >= A) wait_vm<A * WL>(); else wait_units<A - 1, WL>(units);
  }
}

template <int I, int N, class F>
__device__ __forceinline__ void unroll_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    unroll_for<I + 1, N>(f);
  }
}

template <int NX, int CM, bool PRO, int EPI>
__global__ __launch_bounds__(512) void flow_kernel(ProjArgs a, int tiles) {
  constexpr int KW = kFlowWaves, RT = kFlowTile;
  constexpr int MB = (NX + 3) / 4;   // MFMA column blocks of 16 x rows
  constexpr int WL = RT / 4;         // loads per weight unit (4 rows x 256 bytes each)
  constexpr int WS = 16 * RT, XS = 64 * NX;  // 16-byte slots of a weight unit and of an x unit
  constexpr int D = kFlowDepth;  // weight units in flight per wave
  constexpr int XB = flow_x_batch(NX, CM);   // x units staged at once
  constexpr int RW = flow_wave_slots(NX, CM);
  constexpr int OV = (XB * XS + WS - 1) / WS < D ? (XB * XS + WS - 1) / WS : D;  // ring slots under the staged x
  constexpr int BATCHES = (CM + XB - 1) / XB;
  static_assert(D * WL < 64, "vmcnt is 6 bits");
  constexpr int DM = flow_parked(NX, CM, PRO);  // tiles parked before an epilogue
  constexpr int GS = PRO ? 16 * CM : 1;  // gain slots per wave
  __shared__ u32x4_t ring[KW * RW + 256 * MB - XS];  // B operand rows past the loaded ones read on
  __shared__ f32x4_t part[DM][KW][MB][64];
  __shared__ u32x4_t gain[PRO ? KW * GS : 1];
  __shared__ float red[KW][16 * MB];
  __shared__ unsigned long long best_lds[EPI == EPI_ARGMAX ? KW : 1][16];

  const int tid = threadIdx.x, lane = tid & 63;
  const int kw = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, g = lane >> 4;  // MFMA layout: row li, k quarter g
  const int M = a.M, K = a.K, wg = blockIdx.x, G = gridDim.x;
  const int segs = (K + 127) >> 7;
  const int n = (segs - kw + KW - 1) / KW;  // segments of this wave: kw, kw + KW, ... (n <= CM)
  const int my_tiles = (tiles - wg + G - 1) / G;
  const int F = my_tiles * n;               // weight units of this wave

  u32x4_t* const mine = ring + kw * RW;
  int chunk[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) chunk[q] = 8 * ((lane & 15) ^ (4 * g + q));

  // ---- x (and the gain) of this wave's segments, staged through the ring into registers
  const uint16_t* xrow[NX];
#pragma unroll
  for (int q = 0; q < NX; ++q) {
    const int row = 4 * q + g;
    xrow[q] = PRO ? x_row(a, row < M ? row : M - 1) : a.x + (size_t)(row < M ? row : M - 1) * K;
  }
  auto issue_x = [&](int j, int slot) {
    const int k0 = (j * KW + kw) * 128;
#pragma unroll
    for (int q = 0; q < NX; ++q) dma16<0>(xrow[q] + min(k0 + chunk[q & 3], K - 8), mine + slot * XS + 64 * q);
  };
  if constexpr (PRO) {
#pragma unroll
    for (int b = 0; b < (CM + 3) / 4; ++b)
      if (4 * b + g < CM) dma16<0>(a.gamma + min(((4 * b + g) * KW + kw) * 128 + 8 * li, K - 8), gain + kw * GS + 64 * b);
  }
#pragma unroll
  for (int j = 0; j < XB; ++j)
    if (j < n) issue_x(j, j);

  // ---- the weight units, in the order they are used: unit f is segment f % n of step f / n, in
  // ring slot (f + OV) % D: the first D - OV slots lie past the staged x and fill at once, the
  // others when x has been read.
  int wi = 0, wj = 0;                    // step and segment of the next unit to issue
  int wf = 0, wslot = OV == D ? 0 : OV;  // its number and ring slot
  const uint16_t* wrow[WL];
  auto aim = [&]() {
    const int t = ring_tile(wg, wi, G, tiles);
#pragma unroll
    for (int q = 0; q < WL; ++q) wrow[q] = a.w + (size_t)flow_weight_row(EPI, t, 4 * q + g, a.N, RT) * K;
  };
  auto issue_w = [&]() {
    const int k0 = (wj * KW + kw) * 128;
#pragma unroll
    for (int q = 0; q < WL; ++q) dma16<2>(wrow[q] + min(k0 + chunk[q & 3], K - 8), mine + wslot * WS + 64 * q);
    ++wf;
    if (++wslot == D) wslot = 0;
    if (++wj == n) {
      wj = 0;
      ++wi;
      if (wi < my_tiles) aim();
    }
  };
  aim();
#pragma unroll
  for (int f = 0; f < D - OV; ++f)
    if (wf < F) issue_w();

  uint32_t at[4];  // byte offset of this lane's chunk 4 s + g in 16 rows of a unit
#pragma unroll
  for (int s = 0; s < 4; ++s) at[s] = 16 * (li * 16 + ((4 * s + g) ^ ring_swz(li)));
  const uint32_t base = lds_address(mine);

  u32x4_t xr[CM][MB][4];
#pragma unroll
  for (int j = 0; j < CM; ++j)
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int s = 0; s < 4; ++s) xr[j][m][s] = u32x4_t{0u, 0u, 0u, 0u};
  unroll_for<0, BATCHES>([&](auto B) {
    constexpr int b = decltype(B)::value;
    if (b * XB < n) {
      // Newer than the first batch: the weight units issued so far.
      if (b == 0) wait_units<D - OV, WL>(wf); else wait_vm<0>();
      unroll_for<0, XB>([&](auto J) {
        constexpr int j = b * XB + decltype(J)::value;
        if constexpr (j < CM) {
          if (j < n) {
#pragma unroll
            for (int m = 0; m < MB; ++m) {
              uint32_t ax[4];
#pragma unroll
              for (int s = 0; s < 4; ++s) ax[s] = base + at[s] + 16 * ((j - b * XB) * XS + 256 * m);
              read_rows16(ax, xr[j][m]);
            }
          }
        }
      });
#pragma unroll
      for (int j = 0; j < XB; ++j)
        if ((b + 1) * XB + j < n) issue_x((b + 1) * XB + j, j);
    }
  });

#pragma unroll
  for (int f = 0; f < OV; ++f)
    if (wf < F) issue_w();

  // A ragged last segment: nothing past K. Its gain, which may be infinite, is cleared in LDS (it came before
  // x), since operands cleared once more after the norm take 0.5 to 1 % of a launch at up to 8 rows.
  const int tail = (K & 127) && (segs - 1) % KW == kw ? (segs - 1) / KW : -1;  // its unit, or -1
  unroll_for<0, CM>([&](auto J) {
    constexpr int j = decltype(J)::value;
    if (j == tail) {
      const u32x4_t zero = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int s = 0; s < 4; ++s)
        if ((j * KW + kw) * 128 + 32 * s + 8 * g >= K) {
#pragma unroll
          for (int m = 0; m < MB; ++m) xr[j][m][s] = zero;
        }
    }
  });

  // ---- RMSNorm: the rows' sums of squares from the operands, then the operands normalised in place
  if constexpr (PRO) {
    const uint32_t red_at = lds_address(red);
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < CM; ++j)
#pragma unroll
        for (int s = 0; s < 4; ++s) ss = sum_squares8(xr[j][m][s], ss);
      ss += __shfl_xor(ss, 16);
      ss += __shfl_xor(ss, 32);
      if (g == 0) ds_put(red_at + 4 * (kw * 16 * MB + 16 * m + li), ss);
    }
    if (tail >= 0 && g == 0 && (tail * KW + kw) * 128 + 8 * li >= K) {
      const uint32_t to = lds_address(gain) + 16 * (kw * GS + 16 * tail + li);
#pragma unroll
      for (int i = 0; i < 4; ++i) ds_put(to + 4 * i, 0.f);
    }
    lds_barrier();
    float scale[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      static_assert(KW == 8, "ds_sum8");
      const float total = ds_sum8<64 * MB>(red_at + 4 * (16 * m + li));
      scale[m] = 1.0f / sqrtf(total / (float)K + a.eps);
    }
    const uint32_t g_at = lds_address(gain) + 16 * (kw * GS + g);
    unroll_for<0, CM>([&](auto J) {
      constexpr int j = decltype(J)::value;
      u32x4_t gn[4];
      read_gain4(g_at + 256 * j, gn);
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int s = 0; s < 4; ++s) xr[j][m][s] = norm8(xr[j][m][s], gn[s], scale[m]);
    });
  }

  // ---- epilogue of the parked tiles done .. done + count - 1: thread e takes (tile, column block, lane position);
  // lane position 16 gg + ll holds unit rows 4 gg .. 4 gg + 3 of x row 16 m + ll
  unsigned long long best = 0ull;
  auto flush = [&](int count, int done) {
    constexpr int PER = EPI == EPI_SWIGLU ? 32 : 64;  // SwiGLU: the gate positions
    for (int e = tid; e < count * MB * PER; e += 64 * KW) {
      int ln, m, i;
      if constexpr (EPI == EPI_SWIGLU) {
        ln = e & 31, m = (e >> 5) % MB, i = (e >> 5) / MB;
      } else {
        ln = e & 63, m = (e >> 6) % MB, i = (e >> 6) / MB;
      }
      const int ll = (ln & 15) + 16 * m, gg = ln >> 4;
      if (ll >= M || 4 * gg >= (EPI == EPI_SWIGLU ? RT / 2 : RT)) continue;
      const int t = ring_tile(wg, done + i, G, tiles);
      f32x4_t s = part[i][0][m][ln];
#pragma unroll
      for (int w = 1; w < KW; ++w) s += part[i][w][m][ln];
      uint32_t bits[4];
      if constexpr (EPI == EPI_SWIGLU) {
        constexpr int UP = 16 * (RT / 8);  // lane positions from a gate row to its up row
        f32x4_t u = part[i][0][m][ln + UP];
#pragma unroll
        for (int w = 1; w < KW; ++w) u += part[i][w][m][ln + UP];
#pragma unroll
        for (int r = 0; r < 4; ++r) bits[r] = swiglu_bf16(s[r], u[r]);
        const int half = a.N / 2;
        store_row4(a.y + (size_t)ll * half, t * (RT / 2) + 4 * gg, half, bits);
      } else {
        const int n0 = t * RT + 4 * gg;
#pragma unroll
        for (int r = 0; r < 4; ++r) bits[r] = f32_to_bf16(s[r]);
        if (a.y != nullptr) store_row4(a.y + (size_t)ll * a.N, n0, a.N, bits);
        if constexpr (EPI == EPI_ARGMAX) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n0 + r < a.N) best = key_max(best, argmax_key(bf16_to_f32(bits[r]), (uint32_t)(n0 + r)));
        }
      }
    }
  };

  // ---- the walk
  int f = 0, slot = OV == D ? 0 : OV, count = 0, done = 0;
  for (int i = 0; i < my_tiles; ++i) {
    f32x4_t acc[MB] = {};
    unroll_for<0, CM>([&](auto J) {
      constexpr int j = decltype(J)::value;
      if (j < n) {
        wait_units<D - 1, WL>(wf - 1 - f);
        uint32_t aw[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) aw[s] = base + at[s] + 16 * slot * WS;
        u32x4_t w4[4];
        read_rows16(aw, w4);
        if (wf < F) issue_w();
        if (j == tail) {
#pragma unroll
          for (int s = 0; s < 4; ++s)
            if ((j * KW + kw) * 128 + 32 * s + 8 * g >= K) w4[s] = u32x4_t{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int m = 0; m < MB; ++m) acc[m] = mfma16x16x32(w4[s], xr[j][m][s], acc[m]);
        ++f;
        if (++slot == D) slot = 0;
      }
    });
#pragma unroll
    for (int m = 0; m < MB; ++m) part[count][kw][m][lane] = acc[m];
    ++count;
    if (count == DM || i + 1 == my_tiles) {
      lds_barrier();
      flush(count, done);
      done += count;
      count = 0;
      if (i + 1 < my_tiles) lds_barrier();  // the next tiles park in the same slots
    }
  }

  // The rows the norm read (gathered rows), when asked: spread over the grid.
  if constexpr (PRO) {
    if (a.sum != nullptr) {
      const int chunks = K >> 3;
      for (int e = wg * 64 * KW + tid; e < M * chunks; e += G * 64 * KW) {
        const int m = e / chunks, c = e - m * chunks;
        store16(a.sum + (size_t)m * K + 8 * c, load16(x_row(a, m) + 8 * c));
      }
    }
  }
  if constexpr (EPI == EPI_ARGMAX) {
    best = key_max(best, __shfl_xor(best, 16));
    best = key_max(best, __shfl_xor(best, 32));
    if (g == 0) best_lds[kw][li] = best;
    __syncthreads();
    if (tid < M) {
      unsigned long long k = 0ull;
      for (int w = tid >> 4; w < KW; w += MB) k = key_max(k, best_lds[w][tid & 15]);
      a.keys[(size_t)wg * M + tid] = k;
    }
  }
}

typedef void (*FlowKernel)(ProjArgs, int);

template <int NX, int CM, bool PRO>
FlowKernel pick_flow_epilogue(int epi) {
  switch (epi) {
    case EPI_STORE: return flow_kernel<NX, CM, PRO, EPI_STORE>;
    case EPI_SWIGLU: return flow_kernel<NX, CM, PRO, EPI_SWIGLU>;
    case EPI_ARGMAX: return flow_kernel<NX, CM, PRO, EPI_ARGMAX>;
  }
  return nullptr;
}

// Kernel for up to 4 NX x rows and CM segments per wave.
template <int NX, bool PRO>
FlowKernel pick_flow_segments(int c, int epi) {
  if (c <= 1) return pick_flow_epilogue<NX, 1, PRO>(epi);
  if (c <= 2) return pick_flow_epilogue<NX, 2, PRO>(epi);
  if (c <= 3) return pick_flow_epilogue<NX, 3, PRO>(epi);
  if (c <= 4) return pick_flow_epilogue<NX, 4, PRO>(epi);
  if (c <= 5) return pick_flow_epilogue<NX, 5, PRO>(epi);
  return nullptr;
}

}  // namespace ftk
