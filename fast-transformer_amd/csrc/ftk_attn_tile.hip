// The tile kernel of the split-KV decode attention: 16x16x32 BF16 MFMAs fed
// through LDS (ftk_attn.hip holds the launch rule and the merge).
//
// Long caches are bound by HBM reads, short ones by the chain position -> cache
// -> softmax -> merge. A wave takes units of 32 cache slots: direct-to-LDS loads
// bring K and V (64 KB per workgroup at D = 128, so that two fit a CU, no
// registers held), the next K is requested as soon as this one's operands are
// read and the next V as soon as this V's are, so one of the two is in flight
// throughout. K rows are the A operand and the query heads the B operand's
// columns (up to 8 of 16): a lane's four accumulators are one head's scores of
// four slots, so the softmax needs two cross-lane steps per unit. p is already
// in the B operand's layout of the second product, and ds_read_b64_tr_b16 gives
// V's columns as its A operand; p goes in as two BF16 addends of one sign (16
// bits of it, where one rounding keeps 8), since the matrix cores are idle most
// of the time. The cost per unit does not depend on the number of heads: with
// dot products and p V on the VALU it grew with it and passed the loads' time
// from 5 heads per KV head on.
// Measured (partials + merge): 1 x 32K slots, 8 KV heads x 8, 71.1 -> 29.2 us;
// D = 64 x 4 heads 24.4 -> 16.7; 8 x 2K ragged, 8 heads, 39.4 -> 15.2; 16 x 8K
// ragged, 4 heads, 72.9 -> 57.3 (8 intervals); 1 x 32K, 4 heads, 29.9 -> 29.1
// (both before and after with the same intervals).
#include "ftk_attn.h"
#include "ftk_dma.h"

namespace ftk {

namespace {

// K's operands: tile t (slots 16 t .. 16 t + 15 of the unit), step s at at[s] + t * TILE bytes.
template <int S, int TILE>
__device__ __forceinline__ void read_k(const uint32_t (&at)[4], u32x4_t (&k)[2][4]) {
  if constexpr (S == 4) {
    asm volatile(
        "ds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\tds_read_b128 %2, %10\n\tds_read_b128 %3, %11\n\t"
        "ds_read_b128 %4, %8 offset:%12\n\tds_read_b128 %5, %9 offset:%12\n\tds_read_b128 %6, %10 offset:%12\n\t"
        "ds_read_b128 %7, %11 offset:%12\n\ts_waitcnt lgkmcnt(0)"
        : "=&v"(k[0][0]), "=&v"(k[0][1]), "=&v"(k[0][2]), "=&v"(k[0][3]), "=&v"(k[1][0]), "=&v"(k[1][1]),
          "=&v"(k[1][2]), "=&v"(k[1][3])
        : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "n"(TILE)
        : "memory");
  } else {
    static_assert(S == 2, "head dimension 64 or 128");
    asm volatile(
        "ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %4 offset:%6\n\t"
        "ds_read_b128 %3, %5 offset:%6\n\ts_waitcnt lgkmcnt(0)"
        : "=&v"(k[0][0]), "=&v"(k[0][1]), "=&v"(k[1][0]), "=&v"(k[1][1])
        : "v"(at[0]), "v"(at[1]), "n"(TILE)
        : "memory");
  }
}

// V's operands, transposed on the way: four dimension tiles at at[0..3] (32 bytes of 16 rows each),
// slots 4 g .. 4 g + 3 of both slot tiles (v[i][0], v[i][1]). ds_read_b64_tr_b16: of each 16 lanes,
// lane i gives 4 values of row i / 4 from column 4 (i % 4) and receives column i of the four rows.
template <int TILE>
__device__ __forceinline__ void read_v4(const uint32_t* at, u32x2_t (&v)[4][2]) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n\tds_read_b64_tr_b16 %1, %8 offset:%12\n\t"
      "ds_read_b64_tr_b16 %2, %9\n\tds_read_b64_tr_b16 %3, %9 offset:%12\n\t"
      "ds_read_b64_tr_b16 %4, %10\n\tds_read_b64_tr_b16 %5, %10 offset:%12\n\t"
      "ds_read_b64_tr_b16 %6, %11\n\tds_read_b64_tr_b16 %7, %11 offset:%12\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(v[0][0]), "=&v"(v[0][1]), "=&v"(v[1][0]), "=&v"(v[1][1]), "=&v"(v[2][0]), "=&v"(v[2][1]),
        "=&v"(v[3][0]), "=&v"(v[3][1])
      : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "n"(TILE)
      : "memory");
}

// Both halves' (or both 16-lane rows') values beside each other: v_permlane32_swap of v with itself
// gives v[l % 32] and v[l % 32 + 32] in every lane l (v_permlane16_swap: the rows of each pair).
struct Pair {
  float a, b;
};
__device__ __forceinline__ Pair halves(float v) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  const auto p = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return {__uint_as_float(p[0]), __uint_as_float(p[1])};
}
__device__ __forceinline__ Pair row_pairs(float v) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return {__uint_as_float(p[0]), __uint_as_float(p[1])};
}
// Sum, or maximum, over the four lanes li, li + 16, li + 32, li + 48, the same bits in every one of them.
__device__ __forceinline__ float quarter_sum(float v) {
  const Pair r = row_pairs(v);
  const Pair h = halves(r.a + r.b);
  return h.a + h.b;
}
__device__ __forceinline__ float quarter_max(float v) {
  const Pair r = row_pairs(v);
  const Pair h = halves(fmaxf(r.a, r.b));
  return fmaxf(h.a, h.b);
}

// What p's upper 16 bits leave of it, at least the smallest normal number where p is positive. That floor
// adds 2^-126 to weights of up to 1; the largest finite value times it is 4.
__device__ __forceinline__ float low_part(float p) {
  const float rest = p - __uint_as_float(__float_as_uint(p) & 0xFFFF0000u);
  return p > 0.f ? fmaxf(rest, 0x1p-126f) : 0.f;
}

}  // namespace

// ROPE (D = 128): the query heads are normalised and rotated here from the packed QKV row, and the
// split whose interval holds the row's own slot (the position, when it lies inside the cache) takes
// that slot's key and value from the packed row too: it writes them to the cache, reads only the
// slots before it from memory, and starts wave 0's softmax state with the new slot (score s, p = 1).
// No other workgroup of the launch reads that slot.
// (Two waves per SIMD, which the LDS allows at most: without that bound the four-wave builds kept part of
// their state in accumulation registers and moved it back and forth, 1 to 2 % of every call.)
template <int D, int W, bool ROPE>
__global__ __launch_bounds__(64 * W, 2) void attn_tile_kernel(AttnArgs a) {
  constexpr int CH = D / 8;              // 16-byte chunks per cache row
  constexpr int S = D / 32, DT = D / 16;  // MFMA steps of a score, dimension tiles of the numerator
  constexpr int SLOTS = kTileSlots;      // a unit: 32 cache rows of K and of V
  constexpr int RPL = 64 / CH, L = SLOTS / RPL;  // rows per wave load, loads per unit of K (or V)
  constexpr int US = SLOTS * CH;         // 16-byte LDS slots of a unit's K (or V)
  constexpr int TILE = 16 * D * 2;       // bytes of 16 rows
  __shared__ u32x4_t ring[W][2 * US];    // per wave: K, V; at the end the waves' numerators
  __shared__ float m_lds[W][16], l_lds[W][16];
  static_assert(sizeof(ring) >= W * kAttnMaxGroup * D * 4, "the numerators reuse the ring");

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4, G = a.group_size;
  const int group = blockIdx.x / a.splits, split = blockIdx.x - group * a.splits;
  const int row = group / a.kv_heads;
  const int64_t newest = a.position[a.pos_stride * row];
  int64_t shift = 0;  // RoPE phase - position
  if constexpr (ROPE) {
    // One load either way (the position again without phases), in flight beside the position's.
    const int64_t loaded = *(a.phases != nullptr ? a.phases + row : a.position + a.pos_stride * row);
    shift = a.phases != nullptr ? loaded : 0;
  }
  const int64_t seen = newest + 1 < (int64_t)a.capacity ? newest + 1 : (int64_t)a.capacity;
  const int64_t visible = seen > 0 ? seen : 0;
  const int64_t share = interval_slots(a, visible, SLOTS);
  const int64_t begin64 = split * share;
  const int begin = (int)(begin64 < visible ? begin64 : visible);  // an interval past the row is empty
  int end = (int)(begin64 + share < visible ? begin64 + share : visible);
  bool own = ROPE && newest >= begin64 && newest < begin64 + share && newest < (int64_t)a.capacity;
  if (own) end = (int)newest;
  const int units = end > begin ? (end - begin + SLOTS - 1) / SLOTS : 0;

  // ROPE: wave 0 rotates the query heads and wave 1 the key head (lane 4 c + i: chunk c of query head i,
  // or of the key), and both leave them in LDS for everyone. Their loads go out before the cache loads.
  __shared__ u32x4_t head_lds[ROPE ? 6 : 1][16];  // the query heads, the key, the value
  u32x4_t qv[4], x = {0u, 0u, 0u, 0u}, gn = x, cs = x, sn = x, vnew = x;
  if constexpr (ROPE) {
    const int kvh = group - row * a.kv_heads, chunk = lane >> 2, i4 = lane & 3;
    const uint16_t* src = a.packed + (size_t)row * (a.q_heads + 2 * a.kv_heads) * D + chunk * 8;
    // A phase outside the tables reads row 0 instead and writes no slot (the row's output is unspecified).
    const int64_t phase = newest + shift;
    const int64_t at = phase >= 0 && phase < a.table_rows ? phase : 0;
    if (at != phase) own = false;
    if (wave < 2) {
      x = load16(src + (size_t)(wave == 0 ? kvh * G + (i4 < G ? i4 : 0) : a.q_heads + kvh) * D);
      gn = load16((wave == 0 ? a.q_gain : a.k_gain) + chunk * 8);
      cs = load16(a.cos + at * D + chunk * 8);
      sn = load16(a.sin + at * D + chunk * 8);
      vnew = load16(src + (size_t)(a.q_heads + a.kv_heads + kvh) * D);
    }
  } else {
#pragma unroll
    for (int s = 0; s < S; ++s) qv[s] = load16(a.q + ((size_t)group * G + (li < G ? li : 0)) * D + 32 * s + 8 * g);
  }

  // Load q brings rows RPL q + lane / CH of a unit; chunk c of a row goes to place c ^ swz(row). Rows at
  // or past `end` re-read row end - 1 (their scores are -inf and their values zeroed below).
  auto swz = [](int r) { return D == 128 ? ring_swz(r) : (r >> 1) & 7; };
  const size_t cache = (size_t)group * a.capacity * D;
  u32x4_t* const mine = ring[wave];
  auto issue = [&](const uint16_t* base, int unit, u32x4_t* dst) {
    const int first = begin + unit * SLOTS;
#pragma unroll
    for (int q = 0; q < L; ++q) {
      const int r = RPL * q + lane / CH;
      const int t = first + r < end ? first + r : end - 1;
      dma16<2>(base + cache + (size_t)t * D + 8 * ((lane % CH) ^ swz(r)), dst + 64 * q);
    }
  };
  asm volatile("" ::: "memory");
  if (wave < units) {
    issue(a.k, wave, mine);
    issue(a.v, wave, mine + US);
  }

  float m = -INFINITY, l = 0.f;  // head li's maximum, and this lane's share of its denominator
  f32x4_t acc[DT] = {};          // head li's numerators of dimensions 16 i + 4 g .. + 3
  if constexpr (ROPE) {
    u32x4_t knew = x;
    if (wave < 2) {
      knew = quad_head_rope(x, gn, cs, sn, wave == 0 ? a.q_eps : a.k_eps, lane);
      if (wave == 0 || (lane & 3) == 0) head_lds[wave == 0 ? lane & 3 : 4][lane >> 2] = knew;
      if (wave == 1 && (lane & 3) == 0) head_lds[5][lane >> 2] = vnew;
    }
    lds_barrier();
    u32x4_t xk[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      qv[s] = head_lds[li & 3][4 * s + g];
      xk[s] = head_lds[4][4 * s + g];
    }
    if (own && wave == 0) {
      float dot = 0.f;
#pragma unroll
      for (int s = 0; s < 4; ++s) dot = dot8(xk[s], qv[s], dot);
      m = quarter_sum(dot) * a.scale_log2;  // p = exp2(s - s) = 1
      l = g == 0 ? 1.f : 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const u32x2_t v = reinterpret_cast<const u32x2_t*>(head_lds[5])[4 * i + g];
        const uint32_t lo = v[0], hi = v[1];
        acc[i] = f32x4_t{lo_f32(lo), hi_f32(lo), lo_f32(hi), hi_f32(hi)};
      }
    }
    x = knew;
  }
  const u32x4_t zero = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (li >= G) qv[s] = zero;

  uint32_t k_at[4], v_at[8];
  {
    const uint32_t base = lds_address(mine);
#pragma unroll
    for (int s = 0; s < S; ++s) k_at[s] = base + 16 * (li * CH + ((4 * s + g) ^ swz(li)));
    const int r = 4 * g + (li >> 2);  // the row whose values this lane gives to its 16
#pragma unroll
    for (int i = 0; i < DT; ++i)
      v_at[i] = base + 16 * US + 16 * (r * CH + ((2 * i + ((li >> 1) & 1)) ^ swz(r))) + 8 * (li & 1);
  }

  for (int unit = wave; unit < units; unit += W) {
    const int next = unit + W, first = begin + unit * SLOTS;
    const bool more = next < units, ragged = first + SLOTS > end;
    wait_vm<L>();  // K; V may still be in flight
    u32x4_t kr[2][4];
    read_k<S, TILE>(k_at, kr);
    if (more) issue(a.k, next, mine);
    f32x4_t sc[2] = {};
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int t = 0; t < 2; ++t) sc[t] = mfma16x16x32(kr[t][s], qv[s], sc[t]);

    // Element r of sc[t]: slot 16 t + 4 g + r, head li.
    float top = m;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = sc[t][r] * a.scale_log2;
        if (ragged && first + 16 * t + 4 * g + r >= end) v = -INFINITY;
        sc[t][r] = v;
        top = fmaxf(top, v);
      }
    top = quarter_max(top);
    const float pivot = top == -INFINITY ? 0.f : top;
    const float corr = exp2_f32(m - pivot);
    float p[2][4], sum = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[t][r] = exp2_f32(sc[t][r] - pivot);
        sum += p[t][r];
      }
    l = l * corr + sum;
    m = top;
    // p as two BF16 addends, the second product's operands: element e of quarter g is slot 4 g + e of tile 0,
    // then of tile 1. Neither is negative, and where p is not zero neither is zero (low_part): an infinite
    // value then gives that infinity twice over, where 0 x inf or inf - inf would be no number. (Rounding
    // p to nearest and adding what is left with its sign, without that property, takes as long.)
    u32x4_t ph, pl;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const float p0 = p[h >> 1][2 * (h & 1)], p1 = p[h >> 1][2 * (h & 1) + 1];
      ph[h] = __builtin_amdgcn_perm(__float_as_uint(p1), __float_as_uint(p0), 0x07060302u);
      pl[h] = rne_pair(low_part(p0), low_part(p1));
    }
    if (__any(corr != 1.f)) {
#pragma unroll
      for (int i = 0; i < DT; ++i) acc[i] *= corr;
    }

    if (more) wait_vm<L>(); else wait_vm<0>();  // V; the next K may still be in flight
    u32x2_t vr[DT / 4][4][2];
#pragma unroll
    for (int i = 0; i < DT / 4; ++i) read_v4<TILE>(v_at + 4 * i, vr[i]);
    if (more) issue(a.v, next, mine + US);
    if (ragged) {  // values of slots past the end: zero, whatever the re-read row holds
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int slot = first + 16 * t + 4 * g + 2 * h;
          const uint32_t keep = (slot < end ? 0xFFFFu : 0u) | (slot + 1 < end ? 0xFFFF0000u : 0u);
#pragma unroll
          for (int i = 0; i < DT; ++i) vr[i / 4][i % 4][t][h] &= keep;
        }
    }
#pragma unroll
    for (int i = 0; i < DT; ++i) {
      const u32x2_t v0 = vr[i / 4][i % 4][0], v1 = vr[i / 4][i % 4][1];
      const u32x4_t va = {v0[0], v0[1], v1[0], v1[1]};
      acc[i] = mfma16x16x32(va, pl, acc[i]);
      acc[i] = mfma16x16x32(va, ph, acc[i]);
    }
  }

  if constexpr (ROPE) {
    if (own && wave == 1 && (lane & 3) == 0) {
      store16(a.k_store + cache + (size_t)newest * D + (lane >> 2) * 8, x);
      store16(a.v_store + cache + (size_t)newest * D + (lane >> 2) * 8, vnew);
    }
  }

  // The waves' states, merged in wave order (their numerators through the ring's LDS).
  l = quarter_sum(l);
  __syncthreads();  // every wave is past its last read of the ring
  float* const num = reinterpret_cast<float*>(&ring[0][0]);  // [W][G][D]
  if (li < G) {
#pragma unroll
    for (int i = 0; i < DT; ++i)
      *reinterpret_cast<f32x4_t*>(num + ((size_t)wave * G + li) * D + 16 * i + 4 * g) = acc[i];
    if (g == 0) {
      m_lds[wave][li] = m;
      l_lds[wave][li] = l;
    }
  }
  __syncthreads();
  const int t = threadIdx.x;
  if (t < G * CH) {
    const int h = t / CH, cc = t - (t / CH) * CH;
    float mm = m_lds[0][h], ll = l_lds[0][h], aa[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) aa[e] = num[(size_t)h * D + cc * 8 + e];
#pragma unroll
    for (int w = 1; w < W; ++w) {
      float a2[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) a2[e] = num[((size_t)w * G + h) * D + cc * 8 + e];
      merge_state(mm, ll, aa, m_lds[w][h], l_lds[w][h], a2);
    }
    store_state(a, group, split, h, cc, G, D, mm, ll, aa);
  }
}

hipError_t launch_attn_tile(const AttnArgs& a, const AttnShape& s, hipStream_t stream) {
  const dim3 grid((unsigned)(s.groups * s.splits)), block(64 * s.waves);
  const bool rope = a.packed != nullptr;
  if (s.waves != 4 && s.waves != 8) return hipErrorInvalidValue;
  if (s.dim == 128 && rope)
    hipLaunchKernelGGL((s.waves == 4 ? attn_tile_kernel<128, 4, true> : attn_tile_kernel<128, 8, true>), grid, block, 0,
                       stream, a);
  else if (s.dim == 128)
    hipLaunchKernelGGL((s.waves == 4 ? attn_tile_kernel<128, 4, false> : attn_tile_kernel<128, 8, false>), grid, block,
                       0, stream, a);
  else if (s.dim == 64 && !rope)
    hipLaunchKernelGGL((s.waves == 4 ? attn_tile_kernel<64, 4, false> : attn_tile_kernel<64, 8, false>), grid, block, 0,
                       stream, a);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace ftk
