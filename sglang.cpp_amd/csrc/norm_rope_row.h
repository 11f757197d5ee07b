// One head row of a qkv token through qk-RMSNorm and RoPE, in registers: the
// step shared by the fused store pass (rope_norm.hip) and the decode kernel
// that stores its own token (decode.hip), so both write the same bits.
#pragma once

#include "common.h"

namespace sgl {

// One rotated value: x c + p s with the partner's sign applied (p_signed is -p in
// the first half (x c - p s there: negation is exact), as one multiply and
// one fused multiply-add wherever RoPE is applied, so every path rounds
// alike.
__device__ __forceinline__ float rope_one(float x, float p_signed, float c, float s) {
  return fmaf(p_signed, s, x * c);
}

// Sign bits of both 16-bit halves of a packed word (bf16 and fp16 alike).
constexpr uint32_t kSign2 = 0x80008000u;

// The cos/sin values a lane needs: entries [8 jj, 8 jj + 8) of its position's
// row, jj = lane_in_row modulo half the row's LPR lanes.
struct RopeRow {
  f32x4_t c0, c1, s0, s1;
};

__device__ __forceinline__ RopeRow load_rope_row(const float* cos_row, const float* sin_row) {
  RopeRow t;
  t.c0 = *reinterpret_cast<const f32x4_t*>(cos_row);
  t.c1 = *reinterpret_cast<const f32x4_t*>(cos_row + 4);
  t.s0 = *reinterpret_cast<const f32x4_t*>(sin_row);
  t.s1 = *reinterpret_cast<const f32x4_t*>(sin_row + 4);
  return t;
}

// raw: the 8 bf16 values of this lane (LPR lanes hold a row of 8 LPR). Returns
// them normalised by wf (norm), rounded to bf16, rotated and rounded again.
template <int LPR>
__device__ __forceinline__ u32x4_t norm_rope_row(const u32x4_t& raw, bool norm,
                                                 const float (&wf)[8], float eps, bool first,
                                                 const RopeRow& t) {
  constexpr int D = LPR * 8;
  constexpr int HALF = LPR / 2;
  const uint32_t psign = first ? kSign2 : 0u;
  float x[8];
  unpack8(raw, x);
  u32x4_t words = raw;
  if (norm) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) ss += x[i] * x[i];
    ss = group_sum<LPR>(ss);
    const float scale = rsqrtf(ss * (1.0f / D) + eps);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      words[i] = pack_bf16x2((x[2 * i] * scale) * wf[2 * i], (x[2 * i + 1] * scale) * wf[2 * i + 1]);
    unpack8(words, x);
  }
  float p[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t wd = words[i];
    uint32_t pw;
    if constexpr (HALF == 8) pw = dpp_u32<0x128>(wd);
    else pw = static_cast<uint32_t>(__shfl_xor(static_cast<int>(wd), HALF, kWave));
    pw ^= psign;
    p[2 * i] = bf16_lo(pw);
    p[2 * i + 1] = bf16_hi(pw);
  }
  const float c[8] = {t.c0[0], t.c0[1], t.c0[2], t.c0[3], t.c1[0], t.c1[1], t.c1[2], t.c1[3]};
  const float sn[8] = {t.s0[0], t.s0[1], t.s0[2], t.s0[3], t.s1[0], t.s1[1], t.s1[2], t.s1[3]};
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = rope_one(x[i], p[i], c[i], sn[i]);
  return pack8(x);
}

}  // namespace sgl
