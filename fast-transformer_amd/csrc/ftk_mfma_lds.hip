// M = 4..32 skinny BF16 projection, the MFMA kind's default form: one workgroup per
// tile, weight and x segments through a per-wave LDS ring (global_load_lds_dwordx4)
// into 16x16x32 BF16 MFMAs, for any K % 8 == 0 and any N.
//
// Same sums and roundings as the other kinds (engine/kernels/linear.py:50-78
// _skinny_gemm; RMSNorm prologue engine/kernels/rmsnorm.py:21-46; SwiGLU
// engine/kernels/swiglu.py:13-24; greedy argmax engine/kernels/argmax.py:19-48).
//
// What bounds it: HBM for the weights and, past 16 x rows, the x rows every workgroup reads from
// L2 (M / RT times the weight bytes). One tile per workgroup, over all of K: a tile's height is
// chosen so that the tiles fill the CUs once (mfma_lds_default), which also reads x the fewest times.
//
//   * The 128-wide K segments are dealt to KW waves. A wave's unit is one segment: RT weight rows and
//     the x rows, 4 rows x 256 bytes per wave instruction into the RING kind's swizzled layout, DW
//     and XD of them in flight, waited for with exact vmcnts. No barrier before the final sum.
//   * x is streamed beside the weights, so K has no limit and the loop stays small. With the norm each
//     unit is normalised as it is read, after a pre-pass over the x rows: every workgroup pays for
//     both, so FLOW takes the calls with a norm where its registers hold x.
//   * The residual added to the outputs is loaded ahead of the units, not where it is added (four
//     dependent loads at the end otherwise).
//
// us per graph node on MI355X over distinct weights, with the residual add, at 8 / 16 / 24 / 32 rows:
// O 4096 x 4096 8.1 / 8.9 / 9.7 / 10.4, down 4096 x 12288 18.4 / 20.5 / 23.1 / 25.6 (4.4 TB/s at 24;
// the register-fed MFMA kernel took 59 there), 1024 x 2048 4.0 / 4.3 / 4.6 / 5.2 (8.3 before at 8 rows).
#include "ftk_dma.h"
#include "ftk_internal.h"

namespace ftk {

namespace {

// The MFMA operands of one unit, read from the ring and waited for in one block:
// a[t][s] (weight subtile t, K step s) at aw[s] + 4096 t, b[m][s] (x rows 16 m ..
// 16 m + 15) at ax[s] + 4096 m. The compiler would put a wait for every load in
// flight (vmcnt(0)) before a plain read of the ring.
template <int T, int MB>
__device__ __forceinline__ void read_unit(const uint32_t (&aw)[4], const uint32_t (&ax)[4], u32x4_t (&a)[2][4],
                                          u32x4_t (&b)[2][4]) {
  if constexpr (T == 1 && MB == 1) {
    asm volatile(
        "ds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\tds_read_b128 %2, %10\n\tds_read_b128 %3, %11\n\t"
        "ds_read_b128 %4, %12\n\tds_read_b128 %5, %13\n\tds_read_b128 %6, %14\n\tds_read_b128 %7, %15\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[0][2]), "=&v"(a[0][3]), "=&v"(b[0][0]), "=&v"(b[0][1]),
          "=&v"(b[0][2]), "=&v"(b[0][3])
        : "v"(aw[0]), "v"(aw[1]), "v"(aw[2]), "v"(aw[3]), "v"(ax[0]), "v"(ax[1]), "v"(ax[2]), "v"(ax[3])
        : "memory");
  } else if constexpr (T == 1 && MB == 2) {
    asm volatile(
        "ds_read_b128 %0, %12\n\tds_read_b128 %1, %13\n\tds_read_b128 %2, %14\n\tds_read_b128 %3, %15\n\t"
        "ds_read_b128 %4, %16\n\tds_read_b128 %5, %17\n\tds_read_b128 %6, %18\n\tds_read_b128 %7, %19\n\t"
        "ds_read_b128 %8, %16 offset:4096\n\tds_read_b128 %9, %17 offset:4096\n\t"
        "ds_read_b128 %10, %18 offset:4096\n\tds_read_b128 %11, %19 offset:4096\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[0][2]), "=&v"(a[0][3]), "=&v"(b[0][0]), "=&v"(b[0][1]),
          "=&v"(b[0][2]), "=&v"(b[0][3]), "=&v"(b[1][0]), "=&v"(b[1][1]), "=&v"(b[1][2]), "=&v"(b[1][3])
        : "v"(aw[0]), "v"(aw[1]), "v"(aw[2]), "v"(aw[3]), "v"(ax[0]), "v"(ax[1]), "v"(ax[2]), "v"(ax[3])
        : "memory");
  } else if constexpr (T == 2 && MB == 1) {
    asm volatile(
        "ds_read_b128 %0, %12\n\tds_read_b128 %1, %13\n\tds_read_b128 %2, %14\n\tds_read_b128 %3, %15\n\t"
        "ds_read_b128 %4, %12 offset:4096\n\tds_read_b128 %5, %13 offset:4096\n\t"
        "ds_read_b128 %6, %14 offset:4096\n\tds_read_b128 %7, %15 offset:4096\n\t"
        "ds_read_b128 %8, %16\n\tds_read_b128 %9, %17\n\tds_read_b128 %10, %18\n\tds_read_b128 %11, %19\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[0][2]), "=&v"(a[0][3]), "=&v"(a[1][0]), "=&v"(a[1][1]),
          "=&v"(a[1][2]), "=&v"(a[1][3]), "=&v"(b[0][0]), "=&v"(b[0][1]), "=&v"(b[0][2]), "=&v"(b[0][3])
        : "v"(aw[0]), "v"(aw[1]), "v"(aw[2]), "v"(aw[3]), "v"(ax[0]), "v"(ax[1]), "v"(ax[2]), "v"(ax[3])
        : "memory");
  } else {
    static_assert(T == 2 && MB == 2, "operand sets");
    asm volatile(
        "ds_read_b128 %0, %16\n\tds_read_b128 %1, %17\n\tds_read_b128 %2, %18\n\tds_read_b128 %3, %19\n\t"
        "ds_read_b128 %4, %16 offset:4096\n\tds_read_b128 %5, %17 offset:4096\n\t"
        "ds_read_b128 %6, %18 offset:4096\n\tds_read_b128 %7, %19 offset:4096\n\t"
        "ds_read_b128 %8, %20\n\tds_read_b128 %9, %21\n\tds_read_b128 %10, %22\n\tds_read_b128 %11, %23\n\t"
        "ds_read_b128 %12, %20 offset:4096\n\tds_read_b128 %13, %21 offset:4096\n\t"
        "ds_read_b128 %14, %22 offset:4096\n\tds_read_b128 %15, %23 offset:4096\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[0][2]), "=&v"(a[0][3]), "=&v"(a[1][0]), "=&v"(a[1][1]),
          "=&v"(a[1][2]), "=&v"(a[1][3]), "=&v"(b[0][0]), "=&v"(b[0][1]), "=&v"(b[0][2]), "=&v"(b[0][3]),
          "=&v"(b[1][0]), "=&v"(b[1][1]), "=&v"(b[1][2]), "=&v"(b[1][3])
        : "v"(aw[0]), "v"(aw[1]), "v"(aw[2]), "v"(aw[3]), "v"(ax[0]), "v"(ax[1]), "v"(ax[2]), "v"(ax[3])
        : "memory");
  }
}

// The gain's four chunks of one unit for this lane (K steps of 32: 64 bytes apart).
__device__ __forceinline__ void read_gain(uint32_t at, u32x4_t (&g)[4]) {
  asm volatile(
      "ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:64\n\tds_read_b128 %2, %4 offset:128\n\t"
      "ds_read_b128 %3, %4 offset:192\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(g[0]), "=&v"(g[1]), "=&v"(g[2]), "=&v"(g[3])
      : "v"(at)
      : "memory");
}

}  // namespace

template <int NX, int RT, int KW, bool PRO, int EPI>
__global__ __launch_bounds__(64 * KW) void mfma_lds_kernel(ProjArgs a) {
  constexpr int MB = (NX + 3) / 4;       // MFMA column blocks of 16 x rows
  constexpr int T = (RT + 15) / 16;      // MFMA row subtiles (the rows past RT are discarded)
  constexpr int DW = mfma_lds_w_units(RT, KW), XD = mfma_lds_x_units(RT, KW, MB);
  constexpr int WL = RT / 4;             // weight loads per unit (4 rows x 256 bytes each)
  constexpr int WS = 16 * RT, XS = 64 * NX;  // 16-byte slots of a unit's weights and x
  constexpr int RW = mfma_lds_wave_slots(NX, RT, KW);  // slots of one wave's ring
  constexpr int PAD = mfma_lds_pad_slots(NX, RT, KW);  // operand rows past the loaded ones read on
  static_assert(XD <= DW && RW >= 64 * T * MB, "the partials reuse the ring");
  __shared__ u32x4_t ring[KW * RW + PAD];
  __shared__ float red[32];
  __shared__ unsigned long long best_lds[T * MB * 16];
  extern __shared__ u32x4_t gain[];      // PRO: K BF16 rounded up to whole segments

  const int tid = threadIdx.x, lane = tid & 63;
  const int kw = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, g = lane >> 4;  // MFMA layout: row li, k quarter g
  const int M = a.M, K = a.K, tile = blockIdx.x;
  const int segs = (K + 127) >> 7;               // 128-wide K segments; wave kw takes kw, kw + KW, ...
  const int n = (segs - kw + KW - 1) / KW;       // units of this wave (0 for a wave past the segments)

  // ---- where this lane's loads go: load q brings unit row 4 q + lane / 16, chunk swizzled
  int chunk[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) chunk[q] = 8 * ((lane & 15) ^ (4 * g + q));
  const uint16_t* wrow[WL];
#pragma unroll
  for (int q = 0; q < WL; ++q)
    wrow[q] = a.w + (size_t)flow_weight_row(EPI, tile, 4 * q + g, a.N, RT) * K;
  const uint16_t* xrow[NX];
#pragma unroll
  for (int q = 0; q < NX; ++q) {
    const int row = 4 * q + g;
    xrow[q] = PRO ? x_row(a, row < M ? row : M - 1) : a.x + (size_t)(row < M ? row : M - 1) * K;
  }
  u32x4_t* const mine = ring + kw * RW;
  // This thread's outputs of the STORE / ARGMAX epilogue: four rows of subtile kw / MB, x row out_m.
  const int out_m = li + 16 * (kw % MB), out_r = 16 * (kw / MB) + 4 * g, out_n = tile * RT + out_r;
  u32x2_t add = {0u, 0u};
  if constexpr (EPI == EPI_STORE) {
    if (out_r < RT) add = out_add4(a, out_m < M ? out_m : M - 1, out_n);
  }
  auto issue_w = [&](int u, int slot) {
    const int k0 = (u * KW + kw) * 128;
#pragma unroll
    for (int q = 0; q < WL; ++q) dma16<2>(wrow[q] + min(k0 + chunk[q & 3], K - 8), mine + slot * WS + 64 * q);
  };
  auto issue_x = [&](int u, int slot) {
    const int k0 = (u * KW + kw) * 128;
#pragma unroll
    for (int q = 0; q < NX; ++q)
      dma16<0>(xrow[q] + min(k0 + chunk[q & 3], K - 8), mine + DW * WS + slot * XS + 64 * q);
  };
#pragma unroll
  for (int s = -DW; s < 0; ++s) {
    if (s + XD >= 0 && s + XD < n) issue_x(s + XD, s + XD);
    if (s + DW < n) issue_w(s + DW, s + DW);
  }

  // ---- RMSNorm prologue: row scales, and the gain into LDS
  float scale[MB];
  if constexpr (PRO) {
    const int chunks = K >> 3;
    for (int c = tid; c < segs * 16; c += 64 * KW) gain[c] = c < chunks ? load16(a.gamma + 8 * c) : u32x4_t{0u, 0u, 0u, 0u};
    constexpr int RB = (4 * NX + KW - 1) / KW < 4 ? (4 * NX + KW - 1) / KW : 4;  // rows at once
    for (int m0 = kw; m0 < M; m0 += KW * RB) {
      float ss[RB];
      const uint16_t* xr[RB];
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        ss[i] = 0.f;
        xr[i] = x_row(a, m0 + i * KW < M ? m0 + i * KW : m0);
      }
      for (int c0 = lane; c0 < chunks; c0 += 64 * 8) {
        u32x4_t v[RB][8];
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
          for (int j = 0; j < 8; ++j) v[i][j] = load16(xr[i] + 8 * min(c0 + 64 * j, chunks - 1));
#pragma unroll
        for (int i = 0; i < RB; ++i) {
          const int m = m0 + i * KW;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            if (c0 + 64 * j >= chunks) continue;
            ss[i] = sum_squares8(v[i][j], ss[i]);
            if (a.sum != nullptr && tile == 0 && m < M) store16(a.sum + (size_t)m * K + 8 * (c0 + 64 * j), v[i][j]);
          }
        }
      }
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        const float total = wave_sum(ss[i]);
        if (lane == 0 && m0 + i * KW < M) red[m0 + i * KW] = total;
      }
    }
    lds_barrier();
#pragma unroll
    for (int m = 0; m < MB; ++m) scale[m] = li + 16 * m < M ? 1.0f / sqrtf(red[li + 16 * m] / (float)K + a.eps) : 0.f;
  }

  // ---- the units
  uint32_t at[4];  // byte offset of this lane's chunk 4 s + g in a unit's 16 rows
#pragma unroll
  for (int s = 0; s < 4; ++s) at[s] = 16 * (li * 16 + ((4 * s + g) ^ ring_swz(li)));
  const uint32_t w_base = lds_address(mine), x_base = w_base + 16 * DW * WS;
  const uint32_t g_base = lds_address(gain) + 16 * g;
  f32x4_t acc[T][MB] = {};
  // Loads issued after unit u's last one that may still be in flight when it is read.
  constexpr int AHEAD = XD == DW ? (DW - 1) * (NX + WL) : WL + (XD - 1) * (NX + WL);
  for (int u = 0; u < n; ++u) {
    if (u + DW - 1 < n) wait_vm<AHEAD>(); else wait_vm<0>();
    const int ws = u % DW, xs = u % XD;
    uint32_t aw[4], ax[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      aw[s] = w_base + at[s] + 16 * ws * WS;
      ax[s] = x_base + at[s] + 16 * xs * XS;
    }
    u32x4_t w4[2][4], x4[2][4], gn[4];
    if constexpr (PRO) read_gain(g_base + 256 * (u * KW + kw), gn);
    read_unit<T, MB>(aw, ax, w4, x4);
    if (u + XD < n) issue_x(u + XD, xs);
    if (u + DW < n) issue_w(u + DW, ws);
    if constexpr (PRO) {
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int s = 0; s < 4; ++s) x4[m][s] = norm8(x4[m][s], gn[s], scale[m]);
    }
    const int k0 = (u * KW + kw) * 128;
    if (k0 + 128 > K) {  // the ragged last segment: nothing past K
#pragma unroll
      for (int s = 0; s < 4; ++s)
        if (k0 + 32 * s + 8 * g >= K) {
          const u32x4_t zero = {0u, 0u, 0u, 0u};
#pragma unroll
          for (int t = 0; t < T; ++t) w4[t][s] = zero;
#pragma unroll
          for (int m = 0; m < MB; ++m) x4[m][s] = zero;
        }
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int t = 0; t < T; ++t) acc[t][m] = mfma16x16x32(w4[t][s], x4[m][s], acc[t][m]);
  }

  // ---- the waves' partials, summed in wave order (in the ring's LDS)
  lds_barrier();  // every wave is past its last read, and its loads have landed
  f32x4_t* const part = reinterpret_cast<f32x4_t*>(ring);  // [KW][T * MB][64]
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int m = 0; m < MB; ++m) part[(kw * T * MB + t * MB + m) * 64 + lane] = acc[t][m];
  lds_barrier();
  auto total = [&](int e) {  // e = (t MB + m) 64 + lane position
    f32x4_t s = part[e];
#pragma unroll
    for (int w = 1; w < KW; ++w) s += part[w * T * MB * 64 + e];
    return s;
  };

  // ---- epilogue: lane position 16 gg + ll holds tile rows 4 gg .. 4 gg + 3 of x row 16 m + ll
  if constexpr (EPI == EPI_SWIGLU) {
    static_assert(EPI != EPI_SWIGLU || RT == 32, "a gate and an up subtile");
    for (int e = tid; e < 64 * MB; e += 64 * KW) {
      const int ll = (e & 15) + 16 * (e >> 6), gg = (e >> 4) & 3;
      if (ll >= M) continue;
      const f32x4_t gate = total(e), up = total(64 * MB + e);
      const int half = a.N / 2, c0 = tile * 16 + 4 * gg;
      uint16_t* yr = a.y + (size_t)ll * half;
      uint32_t bits[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) bits[r] = swiglu_bf16(gate[r], up[r]);
      store_row4(yr, c0, half, bits);
    }
  } else {
    unsigned long long best = 0ull;
    static_assert(64 * T * MB <= 64 * KW, "one entry per thread");
    if (tid < 64 * T * MB) {
      const f32x4_t s = total(tid);
      const int ll = out_m, n0 = out_n;
      if (ll < M && out_r < RT) {
        uint32_t bits[4];
        store_bits4(a, s, add, bits);
        if (a.y != nullptr) store_row4(a.y + (size_t)ll * a.N, n0, a.N, bits);
        if constexpr (EPI == EPI_ARGMAX) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n0 + r < a.N) best = key_max(best, argmax_key(bf16_to_f32(bits[r]), (uint32_t)(n0 + r)));
        }
      }
      if constexpr (EPI == EPI_ARGMAX) {
        best = key_max(best, __shfl_xor(best, 16));
        best = key_max(best, __shfl_xor(best, 32));
        if (g == 0) best_lds[kw * 16 + li] = best;
      }
    }
    if constexpr (EPI == EPI_ARGMAX) {
      __syncthreads();
      if (tid < M) {
        unsigned long long k = best_lds[tid];
#pragma unroll
        for (int t = 1; t < T; ++t) k = key_max(k, best_lds[t * MB * 16 + tid]);
        a.keys[(size_t)tile * M + tid] = k;
      }
    }
  }
}

// ---- dispatch -------------------------------------------------------------------

typedef void (*MfmaLdsKernel)(ProjArgs);

template <int NX, int RT, int KW>
static MfmaLdsKernel pick_epilogue(int epi, bool pro) {
  if constexpr (!mfma_lds_shape(NX, RT, KW)) {
    return nullptr;
  } else {
    switch (epi) {
      case EPI_STORE:
        return pro ? mfma_lds_kernel<NX, RT, KW, true, EPI_STORE> : mfma_lds_kernel<NX, RT, KW, false, EPI_STORE>;
      case EPI_SWIGLU:
        if constexpr (RT == 32)
          return pro ? mfma_lds_kernel<NX, RT, KW, true, EPI_SWIGLU> : mfma_lds_kernel<NX, RT, KW, false, EPI_SWIGLU>;
        return nullptr;
      case EPI_ARGMAX:
        if constexpr (RT == 16 || RT == 32)
          return pro ? mfma_lds_kernel<NX, RT, KW, true, EPI_ARGMAX> : mfma_lds_kernel<NX, RT, KW, false, EPI_ARGMAX>;
        return nullptr;
    }
    return nullptr;
  }
}

template <int NX>
static MfmaLdsKernel pick_shape(int rt, int kw, int epi, bool pro) {
#define FTK_SHAPE(RT_, KW_) \
  if (rt == RT_ && kw == KW_) return pick_epilogue<NX, RT_, KW_>(epi, pro);
  FTK_SHAPE(8, 8)
  FTK_SHAPE(12, 8)
  FTK_SHAPE(16, 8)
  FTK_SHAPE(20, 8)
  FTK_SHAPE(24, 8)
  FTK_SHAPE(16, 4)
  FTK_SHAPE(24, 4)
  FTK_SHAPE(32, 4)
#undef FTK_SHAPE
  return nullptr;
}

static MfmaLdsKernel pick_mfma_lds(int M, int rt, int kw, int epi, bool pro) {
  if (M < 1 || M > 32) return nullptr;
  switch (flow_x_loads(M)) {
    case 1: return pick_shape<1>(rt, kw, epi, pro);
    case 2: return pick_shape<2>(rt, kw, epi, pro);
    case 4: return pick_shape<4>(rt, kw, epi, pro);
    case 6: return pick_shape<6>(rt, kw, epi, pro);
    default: return pick_shape<8>(rt, kw, epi, pro);
  }
}

bool mfma_lds_supported(int M, int K, int rt, int kw, int epi, bool pro) {
  if (K < 8 || K % 8 || pick_mfma_lds(M, rt, kw, epi, pro) == nullptr) return false;
  return mfma_lds_bytes(flow_x_loads(M), rt, kw, pro ? K : 0) <= 160 * 1024;
}

hipError_t launch_mfma_lds(const ProjArgs& a, int epi, const MfmaLdsShape& s, hipStream_t stream) {
  const bool pro = a.gamma != nullptr;
  if (!mfma_lds_supported(a.M, a.K, s.rows, s.waves, epi, pro) || s.grid != flow_tiles(epi, a.N, s.rows))
    return hipErrorInvalidValue;
  const size_t gain = pro ? (size_t)((a.K + 127) / 128) * 256 : 0;
  hipLaunchKernelGGL(pick_mfma_lds(a.M, s.rows, s.waves, epi, pro), dim3(s.grid), dim3(64 * s.waves), gain, stream, a);
  return hipGetLastError();
}

}  // namespace ftk
