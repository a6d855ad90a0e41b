// Softmax states of the split-KV decode attention, shared by its kernels.
#pragma once

#include "ftk_internal.h"

namespace ftk {

__device__ __forceinline__ float exp2_f32(float x) { return __builtin_amdgcn_exp2f(x); }

// Slots per interval of a row with `visible` slots: the row's own share, in whole steps of `step`
// slots, so every interval has work wherever the row stands in its cache. ceil(visible / splits) by the
// launch's reciprocal (exact below 2^31), because it stands between the position's load and the cache's.
__device__ __forceinline__ int64_t interval_slots(const AttnArgs& a, int64_t visible, int step) {
  const int per = (int)(((uint64_t)((uint32_t)visible + a.splits - 1) * a.split_magic) >> a.split_shift);
  return (int64_t)(per + step - 1) / step * step;
}

// Softmax state (max m, denominator l, numerator a) of one query head over 8 dimensions.
template <int E>
__device__ __forceinline__ void merge_state(float& m, float& l, float (&a)[E], float m2, float l2,
                                            const float (&a2)[E]) {
  const float top = fmaxf(m, m2);
  const float pivot = top == -INFINITY ? 0.f : top;  // nothing seen on either side: keep zeros
  const float c1 = exp2_f32(m - pivot), c2 = exp2_f32(m2 - pivot);
  l = l * c1 + l2 * c2;
#pragma unroll
  for (int e = 0; e < E; ++e) a[e] = a[e] * c1 + a2[e] * c2;
  m = top;
}

// A workgroup's merged state of query head h, dimensions 8 cc .. 8 cc + 7: the
// output itself (one interval) or the interval's FP32 partial and (max, denominator).
__device__ __forceinline__ void store_state(const AttnArgs& a, int group, int split, int h, int cc, int G, int D,
                                            float m, float l, const float (&acc)[8]) {
  if (a.splits == 1) {
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = pack_bf16(acc[2 * i] / l, acc[2 * i + 1] / l);
    store16(a.out + ((size_t)group * G + h) * D + cc * 8, u32x4_t{o[0], o[1], o[2], o[3]});
  } else {
    const size_t slot = ((size_t)group * a.splits + split) * G + h;
    float* dst = a.partial + slot * D + cc * 8;
    *reinterpret_cast<f32x4_t*>(dst) = f32x4_t{acc[0], acc[1], acc[2], acc[3]};
    *reinterpret_cast<f32x4_t*>(dst + 4) = f32x4_t{acc[4], acc[5], acc[6], acc[7]};
    if (cc == 0) *reinterpret_cast<f32x2_t*>(a.stats + slot * 2) = f32x2_t{m, l};
  }
}

// Lane l ^ 32's value: v_permlane32_swap trades lanes 32..63 of its first
// operand with lanes 0..31 of its second; with both = v, the second comes
// back holding v[l + 32] in lanes 0..31 and the first v[l - 32] in lanes 32..63.
__device__ __forceinline__ float lane_xor32(float v, int lane) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  const auto p = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, lane < 32 ? p[1] : p[0]);
}

// Lane l ^ 16's value: v_permlane16_swap trades the odd 16-lane rows of its
// first operand with the even rows of its second.
__device__ __forceinline__ float lane_xor16(float v, int lane) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return __builtin_bit_cast(float, (lane & 16) ? p[0] : p[1]);
}

// Sum over the 16 lanes that share lane bits 0..1, the same bits in all of
// them, on the VALU. row_ror:8 is lane ^ 8 inside a row of 16; its sum is the
// same under ^ 8, so row_ror:4 (which reaches l ^ 4 or l ^ 12) adds lane ^ 4's
// value. Every step adds a lane pair in both orders.
__device__ __forceinline__ float quad_group_sum(float v, int lane) {
  v += dpp<0x128, 0xF>(v);  // row_ror:8
  v += dpp<0x124, 0xF>(v);  // row_ror:4
  v += lane_xor16(v, lane);
  return v + lane_xor32(v, lane);
}

// Head RMSNorm, gain and RoPE of one D = 128 head in the QUAD layout: lane
// 4 c + i holds elements 8 c .. 8 c + 7 (c = 0..15), the 16 lanes of one i the
// whole head; element j + 64 of element j's rotation is in chunk c ^ 8, lane ^ 32.
// n = bf16(x / sqrt(mean(x^2) + eps)), w = bf16(n g),
// out = bf16(bf16(w cos) + bf16(rotate_half(w) sin)) (engine/kernels/qk_rope.py:48-76).
__device__ __forceinline__ u32x4_t quad_head_rope(u32x4_t x, u32x4_t g, u32x4_t c, u32x4_t s, float eps,
                                                  int lane) {
  float xf[8], gf[8], cf[8], sf[8];
  widen8(x, xf);
  widen8(g, gf);
  widen8(c, cf);
  widen8(s, sf);
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) ss += xf[e] * xf[e];
  ss = quad_group_sum(ss, lane);
  const float inv_std = 1.0f / sqrtf(ss / 128.f + eps);
  float w[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) w[e] = round_bf16(round_bf16(xf[e] * inv_std) * gf[e]);
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float r[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int e = 2 * i + j;
      const float partner = lane_xor32(w[e], lane);
      const float rot = lane < 32 ? -partner : partner;  // chunk < 8: the first half of the head
      r[j] = round_bf16(w[e] * cf[e]) + round_bf16(rot * sf[e]);
    }
    o[i] = pack_bf16(r[0], r[1]);
  }
  return u32x4_t{o[0], o[1], o[2], o[3]};
}

constexpr int kTileSlots = 32;  // cache rows in a unit of the tile kernel

// The tile kernel's launch, for any shape (ftk_attn_tile.hip).
hipError_t launch_attn_tile(const AttnArgs& a, const AttnShape& s, hipStream_t stream);

}  // namespace ftk
