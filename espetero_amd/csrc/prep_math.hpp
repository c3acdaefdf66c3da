// The arithmetic of attn_prep for one lane's share of one (row, head), shared by the prep kernel and by
// the streaming attention kernel's fused prologue so that both give the same bits: RMSNorm over the head
// (queries and keys with the learned weight, values without), rotary embedding of the leading rope_dims
// dims in the half-split pairing, the query scale (kernels/40_attention.metal:23-102,
// kernels/80_gemma.metal:63-108, kernels/82_qwen3_omni.metal:39-88).
// A head is HD / 8 consecutive lanes of one wavefront, aligned to that count; every lane of the head must call (the
// norm's sum is a lane exchange). Lane i holds two chunks of 4 consecutive dims: a rotating dim and its partner half the
// rotating dims away, so that the rotation happens inside the lane and reads one (cos, sin) for the two; lanes past the
// rotating dims hold two chunks of the rest. (With 4 consecutive dims per lane the partner came through an LDS exchange
// per dim, and so did the sum: 10 exchanges and 4 table reads per lane and 4 dims at 256 rotating dims, now 0 and 2.)
#pragma once

#include <type_traits>

#include "common.hpp"

namespace esp {

constexpr int kPrepDims = 8;  // dims a lane holds

// First dims of lane li's two chunks.
struct PrepDims {
  int a, b;
  bool rot;  // a and b are partners of the rotation
};
template <int HD>
__device__ __forceinline__ PrepDims prep_dims(const esp_prep_params& p, int li) {
  const int half = p.rope_dims / 2, j = li - half / 4;
  if (j < 0) return {4 * li, 4 * li + half, true};
  return {p.rope_dims + 4 * j, p.rope_dims + 4 * j + (HD - p.rope_dims) / 2, false};
}

// The sum of v over the LPH lanes of a head, in every one of them: rotations inside a row of 16 lanes, then whole rows
// exchanged. a + b == b + a, so all lanes of a head end on the same bits.
template <int LPH>
__device__ __forceinline__ float prep_head_sum(float v) {
#pragma clang fp contract(off)
  auto ror = [](float x, auto by) __attribute__((always_inline)) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 + decltype(by)::value, 0xf, 0xf, true));
  };
  v += ror(v, std::integral_constant<int, 8>{});
  v += ror(v, std::integral_constant<int, 4>{});
  v += ror(v, std::integral_constant<int, 2>{});
  v += ror(v, std::integral_constant<int, 1>{});
  // (the results as scalars first: a bit cast of a vector's element takes the vector's first one here)
  if constexpr (LPH >= 32) {
    const auto w = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
    const uint32_t even = w[0], odd = w[1];
    v = __builtin_bit_cast(float, even) + __builtin_bit_cast(float, odd);
  }
  if constexpr (LPH >= 64) {
    const auto w = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
    const uint32_t low = w[0], high = w[1];
    v = __builtin_bit_cast(float, low) + __builtin_bit_cast(float, high);
  }
  return v;
}

// x: the lane's dims of the fp32 projection (chunk a, then chunk b), rewritten in place. kind: 0 query, 1 key, 2 value.
// w: the norm weight of those dims (1 for values). cs: (cos, sin) per frequency of this row; li: the lane's place in its
// head. No branches: a caller's rows interleave.
template <int HD>
__device__ __forceinline__ void prep_lane(float (&x)[kPrepDims], int kind, const float (&w)[kPrepDims], const float2* cs,
                                          const esp_prep_params& p, int li, bool rot) {
  // Two kernels inline this function and must agree to the bit, so nothing here is left to the compiler's
  // choice of which multiply to fuse with which add: the fused operations are spelled out, the rest stays apart.
#pragma clang fp contract(off)
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < kPrepDims; ++i) ss = __builtin_fmaf(x[i], x[i], ss);
  ss = prep_head_sum<HD / kPrepDims>(ss);
  float inv = rsqrtf(ss / float(HD) + p.eps);
  asm volatile("" : "+v"(inv));  // worked out in every lane, not under a branch
  inv = (kind != 2 || p.v_norm) ? inv : 1.0f;
#pragma unroll
  for (int i = 0; i < kPrepDims; ++i) x[i] = x[i] * inv * w[i];
  const bool turn = rot && kind != 2;
  const float scale = kind == 0 ? p.q_scale : 1.0f;
  const float4* t4 = reinterpret_cast<const float4*>(cs + (rot ? 4 * li : 0));  // chunk a starts at frequency 4 li
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float4 t2 = t4[i / 2];
    const float c = i % 2 ? t2.z : t2.x, sn = i % 2 ? t2.w : t2.y;
    const float lo = x[i], hi = x[4 + i];
    const float lo_turn = hi * sn, hi_turn = lo * sn;
    x[i] = (turn ? __builtin_fmaf(lo, c, -lo_turn) : lo) * scale;
    x[4 + i] = (turn ? __builtin_fmaf(hi, c, hi_turn) : hi) * scale;
  }
}

// (cos, sin) of a row's rotation angle: a frequency turns by position component sel times freq.
__device__ __forceinline__ float2 prep_cos_sin(const int4 pr, int sel, float freq) {
  const float position = float(sel == 0 ? pr.x : (sel == 1 ? pr.y : pr.z));
  float sn, c;
  sincosf(position * freq, &sn, &c);
  return make_float2(c, sn);
}

// 4 dims (d ..) of one key or value row, as stored, into position ps of the pool block whose head starts at hb. (V lies
// transposed there: an element store per dim.)
template <int HD>
__device__ __forceinline__ void prep_append(uint16_t* hb, int kind, int bt, int ps, int d, u32x2 v) {
  if (kind == 1) {
    *reinterpret_cast<u32x2*>(hb + size_t(ps) * HD + d) = v;
    return;
  }
  uint16_t* vt = hb + vt_elem(bt, HD, ps, d);
#pragma unroll
  for (int i = 0; i < 4; ++i) vt[i * kVtDim] = uint16_t(v[i / 2] >> (16 * (i & 1)));
}

}  // namespace esp
