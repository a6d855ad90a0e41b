// Q/K head RMSNorm, RoPE and the KV-cache update of one decode (or prefill)
// step on gfx950: engine/kernels/qk_rope.py:13-94 (_qk_rope_cache).
//
// Two forms of one arithmetic: qk_rope_kernel (FP32 partials, or pointers that
// are not 16-byte aligned, or few heads of 64) gives one wave to a (row, head);
// qk_rope_rows_kernel gives D / 8 lanes to a head. Arithmetic is FP32
// with the reference's roundings: n = bf16(x inv_std), w = bf16(n gain),
// out = bf16(bf16(w cos) + bf16(rot sin)). Query heads go to the token-major
// query [rows, Hq, D]; key heads and the copied value heads to the caches
// [B, Hkv, C, D] at the step's slot. Slots outside the cache and table phases
// outside the cos/sin tables (device-side values the host cannot check) are
// skipped: nothing is read or written out of bounds.
#include "../../include/ftk.h"
#include "ftk_internal.h"

namespace ftk {

template <int E>
__device__ __forceinline__ void load_merged(const RopeArgs& a, int64_t at, float (&v)[E]) {
  if (a.splits == 1) {
    const uint16_t* p = reinterpret_cast<const uint16_t*>(a.packed) + at;
    if constexpr (E == 2) {
      const uint32_t pair = *reinterpret_cast<const uint32_t*>(p);
      v[0] = lo_f32(pair);
      v[1] = hi_f32(pair);
    } else {
      v[0] = bf16_to_f32(*p);
    }
    return;
  }
  const float* p = reinterpret_cast<const float*>(a.packed) + at;
#pragma unroll
  for (int e = 0; e < E; ++e) v[e] = p[e];
  for (int s = 1; s < a.splits; ++s)
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] += p[(size_t)s * a.split_stride + e];
#pragma unroll
  for (int e = 0; e < E; ++e) v[e] = round_bf16(v[e]);
}

template <int E>
__device__ __forceinline__ void store_bf16(uint16_t* p, const float (&v)[E]) {
  if constexpr (E == 2) {
    *reinterpret_cast<uint32_t*>(p) = pack_bf16(v[0], v[1]);
  } else {
    *p = (uint16_t)f32_to_bf16(v[0]);
  }
}

template <int E>
__device__ __forceinline__ void load_table(const uint16_t* p, float (&v)[E]) {
  if constexpr (E == 2) {
    const uint32_t pair = *reinterpret_cast<const uint32_t*>(p);
    v[0] = lo_f32(pair);
    v[1] = hi_f32(pair);
  } else {
    v[0] = bf16_to_f32(*p);
  }
}

// One wave per (row, head), W heads of one row to a workgroup. Lane l holds the
// D / 64 consecutive elements starting at l D / 64, so the RoPE partner of each
// element (D / 2 away) sits in lane l ^ 32: one shuffle.
template <int D, int W>
__global__ __launch_bounds__(64 * W) void qk_rope_kernel(RopeArgs a) {
  constexpr int E = D / 64;
  const int lane = threadIdx.x & 63;
  const int head = blockIdx.y * W + (threadIdx.x >> 6);
  const int heads = a.q_heads + a.kv_heads;
  if (head >= heads) return;  // no barrier in this kernel
  const int r = blockIdx.x;  // row = b * tokens + t
  const int b = r / a.tokens, t = r - b * a.tokens;
  const int col = lane * E;
  const int64_t np = (int64_t)(a.q_heads + 2 * a.kv_heads) * D;
  const bool is_q = head < a.q_heads;

  // Every load that does not depend on the device-side position goes out first
  // (one memory round trip); with shared or per-row cos/sin rows the phase is
  // the token or the row, checked against the tables on the host.
  const bool table = (a.mode & FTK_ROPE_TABLE) != 0;
  const int64_t vat = r * np + (int64_t)(a.q_heads + a.kv_heads + (head - a.q_heads)) * D + col;
  float x[E], g[E], c[E], s[E];
  uint32_t vbits = 0;
  load_merged<E>(a, r * np + (int64_t)head * D + col, x);
  load_table<E>((is_q ? a.q_gain : a.k_gain) + col, g);
  if (!is_q && a.splits == 1) {
    const uint16_t* src = reinterpret_cast<const uint16_t*>(a.packed) + vat;
    vbits = E == 2 ? *reinterpret_cast<const uint32_t*>(src) : (uint32_t)*src;
  }
  int64_t phase = (a.mode & FTK_ROPE_ROWS) ? r : t;
  if (!table) {
    load_table<E>(a.cos + phase * D + col, c);
    load_table<E>(a.sin + phase * D + col, s);
  }
  int64_t slot = 0;
  if (!is_q) slot = (a.mode & FTK_ROPE_PREFILL) ? t : a.position[(a.mode & FTK_ROPE_ROWS) ? b : 0] + t;
  if (table) {
    phase = a.position[b] + a.phases[r];
    if (phase < 0 || phase >= a.table_rows) return;  // wave-uniform; no barrier in this kernel
    load_table<E>(a.cos + phase * D + col, c);
    load_table<E>(a.sin + phase * D + col, s);
  }

  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < E; ++e) ss += x[e] * x[e];
  ss = wave_sum(ss);
  const float inv_std = 1.0f / sqrtf(ss / (float)D + (is_q ? a.q_eps : a.k_eps));
  float w[E], out[E];
#pragma unroll
  for (int e = 0; e < E; ++e) w[e] = round_bf16(round_bf16(x[e] * inv_std) * g[e]);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const float partner = __shfl_xor(w[e], 32);  // element col + D/2 (mod D)
    const float rot = lane < 32 ? -partner : partner;
    out[e] = round_bf16(w[e] * c[e]) + round_bf16(rot * s[e]);
  }
  if (is_q) {
    store_bf16<E>(a.query + ((int64_t)r * a.q_heads + head) * D + col, out);
    return;
  }
  if (slot < 0 || slot >= a.capacity) return;
  const int kv = head - a.q_heads;
  const int64_t at = (((int64_t)b * a.kv_heads + kv) * a.capacity + slot) * D + col;
  store_bf16<E>(a.keys + at, out);
  if (a.splits == 1) {  // the value head as it is, bit for bit
    if constexpr (E == 2) {
      *reinterpret_cast<uint32_t*>(a.values + at) = vbits;
    } else {
      a.values[at] = (uint16_t)vbits;
    }
  } else {
    float v[E];
    load_merged<E>(a, vat, v);
    store_bf16<E>(a.values + at, v);
  }
}

// The pair of lane l ^ (LANES / 2) of each group of LANES lanes (16 or 8). row_ror:8 is l ^ 8 within 16
// lanes; row_half_mirror (7 - l) and then quad_perm [3,2,1,0] (l ^ 3) together are l ^ 4 within 8.
template <int LANES>
__device__ __forceinline__ uint32_t half_partner(uint32_t v) {
  if constexpr (LANES == 16) return dpp_u32<0x128, 0xF>(v);
  return dpp_u32<0x1B, 0xF>(dpp_u32<0x141, 0xF>(v));
}

// Sum over each group of LANES lanes, the same bits in all of them. For 16 lanes the order of the chunks
// is quad_group_sum's (^ 2, ^ 1, ^ 4, ^ 8), so a head is scaled as the fused attention prologue scales it.
template <int LANES>
__device__ __forceinline__ float head_sum(float v) {
  v += dpp<0x4E, 0xF>(v);   // quad_perm [2,3,0,1]: ^ 2
  v += dpp<0xB1, 0xF>(v);   // quad_perm [1,0,3,2]: ^ 1
  v += dpp<0x141, 0xF>(v);  // row_half_mirror: the other four of the eight
  if constexpr (LANES == 16) v += dpp<0x128, 0xF>(v);
  return v;
}

// BF16 rows on 16-byte aligned pointers: D / 8 lanes hold a head, 16 bytes each; a workgroup takes
// 2 ^ log_rows rows and, of each, up to U x (its head groups per row) heads, every row's heads (values
// included) in memory order, so a wave reads 1 KB contiguous. cos, sin and the gains are widened once per
// row and serve its U heads; all loads of a thread go out together. A prompt is bound by the copy's
// traffic once the lanes carry 8 elements: with 2 (one wave per head) the address, table and shuffle
// work per element was the bound. 4000 rows of 32 + 8 + 8 heads of 128 (98 MB): 53.3 -> 24.8 us.
template <int D, int U>
__global__ __launch_bounds__(kThreads) void qk_rope_rows_kernel(RopeArgs a, int rows, int log_rows) {
  constexpr int LANES = D / 8, GROUPS = kThreads / LANES;
  const int lane = threadIdx.x & (LANES - 1), group = (int)threadIdx.x / LANES;
  const int per_row = GROUPS >> log_rows;  // head groups of one row
  const int64_t row = ((int64_t)blockIdx.x << log_rows) + group / per_row;
  if (row >= rows) return;  // whole groups; no barrier in this kernel
  const int r = (int)row;
  const int b = r / a.tokens, t = r - b * a.tokens;
  const int heads = a.q_heads + 2 * a.kv_heads;
  const int first = (int)blockIdx.y * per_row * U + (group & (per_row - 1));
  const int col = lane * 8;

  const uint16_t* src = reinterpret_cast<const uint16_t*>(a.packed) + (int64_t)r * heads * D + col;
  u32x4_t x[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int h = first + u * per_row;
    x[u] = load16(src + (int64_t)(h < heads ? h : heads - 1) * D);
  }
  const u32x4_t qg = load16(a.q_gain + col), kg = load16(a.k_gain + col);
  const bool table = (a.mode & FTK_ROPE_TABLE) != 0;
  int64_t phase = (a.mode & FTK_ROPE_ROWS) ? r : t;
  int64_t slot = t;
  if (!(a.mode & FTK_ROPE_PREFILL)) slot += a.position[(a.mode & FTK_ROPE_ROWS) ? b : 0];
  if (table) {
    phase = a.position[b] + a.phases[r];
    if (phase < 0 || phase >= a.table_rows) return;
  }
  const u32x4_t cw = load16(a.cos + phase * D + col), sw = load16(a.sin + phase * D + col);
  float cf[8], sf[8];
  widen8(cw, cf);
  // The first half of a head takes minus its partner: the sign goes into sin, once.
  const uint32_t flip = lane < LANES / 2 ? 0x80008000u : 0u;
  const uint32_t s0 = sw[0], s1 = sw[1], s2 = sw[2], s3 = sw[3];
  widen8(u32x4_t{s0 ^ flip, s1 ^ flip, s2 ^ flip, s3 ^ flip}, sf);

#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int h = first + u * per_row;
    if (h >= heads) return;
    const int kv = h - a.q_heads, vh = kv - a.kv_heads;
    if (kv >= 0 && (slot < 0 || slot >= a.capacity)) return;  // the heads after it are cache heads too
    const int64_t at = kv < 0 ? ((int64_t)r * a.q_heads + h) * D + col
                              : (((int64_t)b * a.kv_heads + (vh < 0 ? kv : vh)) * a.capacity + slot) * D + col;
    if (vh >= 0) {  // the value head as it is, bit for bit
      store16(a.values + at, x[u]);
      continue;
    }
    float xf[8];
    widen8(x[u], xf);
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += xf[e] * xf[e];
    ss = head_sum<LANES>(ss);
    const float inv_std = 1.0f / sqrtf(ss / (float)D + (kv < 0 ? a.q_eps : a.k_eps));
    float gf[8];
    widen8(kv < 0 ? qg : kg, gf);
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t n = rne_pair(xf[2 * i] * inv_std, xf[2 * i + 1] * inv_std);
      const uint32_t w = rne_pair(lo_f32(n) * gf[2 * i], hi_f32(n) * gf[2 * i + 1]);
      const uint32_t p = half_partner<LANES>(w);
      const uint32_t wc = rne_pair(lo_f32(w) * cf[2 * i], hi_f32(w) * cf[2 * i + 1]);
      const uint32_t ps = rne_pair(lo_f32(p) * sf[2 * i], hi_f32(p) * sf[2 * i + 1]);
      o[i] = pack_bf16(lo_f32(wc) + lo_f32(ps), hi_f32(wc) + hi_f32(ps));
    }
    store16((kv < 0 ? a.query : a.keys) + at, u32x4_t{o[0], o[1], o[2], o[3]});
  }
}

namespace {

// Few heads of 64 stay with the general form: a launch of a few workgroups is one chain of loads and sums, and
// with eight elements to a lane it is the longer one. us, general / rows form: 1 x 18 heads 2.1 / 2.3, 32 x 18
// 2.3 / 2.5, 16 x 80 2.4 / 2.5, 128 x 18 2.5 / 2.6, 64 x 48 2.6 / 2.6, 64 x 80 3.0 / 2.6, 1024 x 80 16.9 / 7.9.
// Heads of 128 are as fast or faster in the rows form throughout (1 x 6 2.2 / 2.2, 32 x 48 2.5 / 2.5).
constexpr int64_t kFewHeads64 = 2560;

bool rows_form(const RopeArgs& a, int rows) {
  const void* ptrs[] = {a.packed, a.q_gain, a.k_gain, a.cos, a.sin, a.query, a.keys, a.values};
  for (const void* p : ptrs)
    if (reinterpret_cast<uintptr_t>(p) & 15u) return false;
  return a.splits == 1 && (a.dim == 128 || (int64_t)rows * (a.q_heads + 2 * a.kv_heads) >= kFewHeads64);
}

template <int D>
hipError_t launch_rows(const RopeArgs& a, int rows, hipStream_t stream) {
  constexpr int GROUPS = kThreads * 8 / D;
  const int heads = a.q_heads + 2 * a.kv_heads;
  int log_rows = 0;  // few heads (one GPU's share of a model): several rows to a workgroup
  while ((GROUPS >> (log_rows + 1)) >= heads) ++log_rows;
  const int per_row = GROUPS >> log_rows;
  const int passes = (heads + per_row - 1) / per_row;
  const unsigned blocks = (unsigned)(((int64_t)rows + (1 << log_rows) - 1) >> log_rows);
  // Heads of a row stay in one workgroup only where the rows alone fill the CUs several times over.
  const int u = blocks < 1024 ? 1 : passes < 4 ? passes : 4;
  typedef void (*Kernel)(RopeArgs, int, int);
  static const Kernel kernels[4] = {qk_rope_rows_kernel<D, 1>, qk_rope_rows_kernel<D, 2>, qk_rope_rows_kernel<D, 3>,
                                    qk_rope_rows_kernel<D, 4>};
  hipLaunchKernelGGL(kernels[u - 1], dim3(blocks, (unsigned)((passes + u - 1) / u)), dim3(kThreads), 0, stream, a,
                     rows, log_rows);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_qk_rope(const RopeArgs& a, int rows, hipStream_t stream) {
  if (rows_form(a, rows)) return a.dim == 128 ? launch_rows<128>(a, rows, stream) : launch_rows<64>(a, rows, stream);
  constexpr int W = 4;
  const dim3 grid((unsigned)rows, (unsigned)((a.q_heads + a.kv_heads + W - 1) / W));
  if (a.dim == 128)
    hipLaunchKernelGGL((qk_rope_kernel<128, W>), grid, dim3(64 * W), 0, stream, a);
  else
    hipLaunchKernelGGL((qk_rope_kernel<64, W>), grid, dim3(64 * W), 0, stream, a);
  return hipGetLastError();
}

}  // namespace ftk
