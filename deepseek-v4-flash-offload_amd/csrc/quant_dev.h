// Per-thread bodies of the activation quantisers, shared by the standalone
// kernels (quant.hip) and the fused align + quantise launch (align.hip).
// One thread owns 8 consecutive bf16 elements (group g); the lanes of one
// quantisation block are consecutive lanes of one wave (16 lanes per 128-element
// FP8 block, 4 lanes per 32-element MXFP4 block), so the block's amax is a
// reduction over one DPP row (quad). The caller maps lanes to groups so that g % 16
// (resp. g % 4) equals the lane's position in its block.
#pragma once
#include "common.h"

namespace dsv4 {

// two floats -> packed bf16 (RNE, NaN -> 0x7fc0 as f32_to_bf16), low half = a;
// cvt_pk_bf16: the converter alone, which keeps a NaN's sign and payload
DSV4_DEV uint32_t cvt_pk_bf16(float a, float b) {
  typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, v2bf{(__bf16)a, (__bf16)b});
}
DSV4_DEV uint32_t pk_bf16(float a, float b) {
  const uint32_t w = cvt_pk_bf16(a, b);
  return (a != a ? 0x7fc0u : w & 0xffffu) | (b != b ? 0x7fc00000u : w & 0xffff0000u);
}
DSV4_DEV float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
DSV4_DEV float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// silu(min(g, L)) * clamp(u, +-L) * w for bf16-rounded g, u (deepseek_v4.py:184-187),
// the one formula of every gate/up epilogue: a token row gets the same h whichever
// kernel its expert runs on. limit <= 0: no clamps.
DSV4_DEV float swiglu(float gt, float up, float w, float limit) {
  if (limit > 0.0f) {
    up = fminf(fmaxf(up, -limit), limit);
    gt = fminf(gt, limit);
  }
  return gt / (1.0f + expf(-gt)) * up * w;
}

// act_quant (npu_ops.py:73-104): per-128 block of one row,
//   amax = max(max|x|, 1e-4); s = 2^ceil(log2(max(amax * fp32(1/448), 2^-126)))
//   code = e4m3fn(clamp(x / s, +-448)) (RNE); rt = bf16(e4m3(code) * s)
// block exponent k of a 128-element FP8 block with abs-max amax (scale 2^k)
DSV4_DEV int fp8_block_exp(float amax) {
  amax = fmaxf(amax, 1e-4f);
  float vs = fmaxf(amax * (1.0f / 448.0f), 1.1754943508222875e-38f);
  return ceil_log2(vs);
}

// Largest value over the 16 lanes of a DPP row (the lanes of one FP8 block), in all of
// them; quad_max: over 4 consecutive lanes (one MXFP4 block). Lane permutes inside the
// VALU: a shuffle through the LDS crossbar per step was the longest chain of a quantiser.
template <int CTRL>
DSV4_DEV float dpp_max(float v) {
  return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false)));
}
DSV4_DEV float quad_max(float v) { return dpp_max<0x4e>(dpp_max<0xb1>(v)); }  // quad_perm xor 1, xor 2
DSV4_DEV float row16_max(float v) { return dpp_max<0x140>(dpp_max<0x141>(quad_max(v))); }  // half-row, row mirror

// E4M3fn codes of f[0..3] times inv = 2^-k, byte 0 first: the clamp of act_quant, then
// the hardware converter, which rounds to nearest even as torch's cast does (the same
// code as the former integer rounding for every fp32 in +-448; the clamp maps NaN to -448).
DSV4_DEV uint32_t fp8_codes4(const float* f, float inv) {
  float y[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) y[i] = fminf(fmaxf(f[i] * inv, -448.0f), 448.0f);
  const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], 0, false);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], lo, true);
}
// 8 bf16 of one 16-byte load as floats; returns their largest magnitude
DSV4_DEV float unpack8(const uint4 v, float* f) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = bf16_to_f32(w[i] & 0xffffu);
    f[2 * i + 1] = bf16_to_f32(w[i] >> 16);
    amax = fmaxf(amax, fmaxf(fabsf(f[2 * i]), fabsf(f[2 * i + 1])));
  }
  return amax;
}

// Group g (already loaded: v) of a tensor; `live` must be the same for the 16 lanes of a block.
DSV4_DEV void fp8_quant_loaded(const uint4 v, int64_t g, bool live, uint4* __restrict__ rt, uint2* __restrict__ codes,
                               float* __restrict__ scale_f32, uint32_t* __restrict__ scale_e8m0x4) {
  float f[8];
  const float amax = row16_max(unpack8(v, f));
  const int k = fp8_block_exp(amax);
  const float inv = pow2f(-k);
  const uint2 c = make_uint2(fp8_codes4(f, inv), fp8_codes4(f + 4, inv));
  if (!live) return;
  if (rt) {  // code * 2^k has at most 4 significant bits, so the upper half of the fp32 is the bf16
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const float s = pow2f(k);
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int w = (int)(i < 2 ? c.x : c.y);
      const f32x2 q = (i & 1) ? __builtin_amdgcn_cvt_pk_f32_fp8(w, true) : __builtin_amdgcn_cvt_pk_f32_fp8(w, false);
      o[i] = (__float_as_uint(q.x * s) >> 16) | (__float_as_uint(q.y * s) & 0xffff0000u);
    }
    rt[g] = make_uint4(o[0], o[1], o[2], o[3]);
  }
  if (codes) codes[g] = c;
  if ((g & 15) == 0) {
    const int64_t blk = g >> 4;
    if (scale_f32) scale_f32[blk] = pow2f(k);
    if (scale_e8m0x4) scale_e8m0x4[blk] = (uint32_t)(k + 127) * 0x01010101u;
  }
}

// A workgroup's share of a tensor: U groups per thread, NT apart (consecutive lanes on
// consecutive groups), from group `wg` * U * NT on; every load is issued before the first
// is used. n_groups is a multiple of 16, so a block's lanes are live together.
template <int U, int NT>
DSV4_DEV void fp8_quant_wg(const uint4* __restrict__ x, int64_t wg, int64_t n_groups, uint4* __restrict__ rt,
                           uint2* __restrict__ codes, float* __restrict__ scale_f32,
                           uint32_t* __restrict__ scale_e8m0x4) {
  const int64_t g0 = wg * (U * NT) + threadIdx.x;
  uint4 v[U];
#pragma unroll
  for (int i = 0; i < U; ++i) v[i] = g0 + i * NT < n_groups ? x[g0 + i * NT] : make_uint4(0, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < U; ++i)
    fp8_quant_loaded(v[i], g0 + i * NT, g0 + i * NT < n_groups, rt, codes, scale_f32, scale_e8m0x4);
}

// MXFP4 activation quant, per 32 elements.
//  rule 0 "ceil_div6" (npu_ops.py:107-121):
//     amax = max(max|x|, 6*2^-126); s = 2^ceil(log2(max(amax*fp32(1/6), 2^-126)))
//     v = clamp(x/s, +-6); q = E2M1-RNE(|v|); sign = (v < 0); dq = bf16(+-q * s)
//  rule 1 "ocp_floor" (OCP MX v1.0): shared = floor(log2 amax) - 2 clamped to
//     [-127, 127] (-127 for an all-zero block); q = E2M1-RNE(min(|x|/2^shared, 6));
//     sign = signbit(x)
// Outputs: packed nibbles (low = even element), E8M0 scale byte, optional bf16 dq.
// shared exponent of an MXFP4 block with abs-max `amax` (rule 0 / 1 as above)
DSV4_DEV int mxfp4_block_exp(float amax, int rule) {
  if (rule == 0) {
    amax = fmaxf(amax, 6.0f * 1.1754943508222875e-38f);
    float vs = fmaxf(amax * (1.0f / 6.0f), 1.1754943508222875e-38f);
    return ceil_log2(vs);
  }
  return (amax == 0.0f) ? -127 : min(max(floor_log2(amax) - 2, -127), 127);
}

// Two floats already in [-6, 6] as sign-magnitude E2M1 nibbles in byte SEL of `old` (low
// nibble = a): the hardware converter (round to nearest even, the sign of the input).
template <int SEL>
DSV4_DEV uint32_t e2m1_pair(uint32_t old, float a, float b) {
  return __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(old, a, b, 1.0f, SEL);
}

// Element f times inv = 2^-k clamped to the E2M1 range, with the sign its nibble takes:
// rule 0 the sign of the clamped quotient (NaN clamps to -6), +0 for either zero; rule 1
// the sign bit of f.
DSV4_DEV float mxfp4_clamped(float f, float inv, int rule) {
  if (rule == 0) return fminf(fmaxf(f * inv, -6.0f), 6.0f) + 0.0f;  // -0 + 0 = +0
  return copysignf(fminf(fabsf(f * inv), 6.0f), f);
}
// the same for f that is not NaN, one instruction shorter under rule 1
DSV4_DEV float mxfp4_clamped_number(float f, float inv, int rule) {
  const float y = fminf(fmaxf(f * inv, -6.0f), 6.0f);
  return rule == 0 ? y + 0.0f : y;
}

// Group g (already loaded: v) of a tensor; `live` must be the same for the 4 lanes of a block.
DSV4_DEV void mxfp4_quant_loaded(const uint4 v, int64_t g, bool live, int rule, uint32_t* __restrict__ packed,
                                 uint8_t* __restrict__ scale, uint4* __restrict__ dq) {
  float f[8];
  const float amax = quad_max(unpack8(v, f));
  const int k = mxfp4_block_exp(amax, rule);
  const float inv = pow2f(-k);
  if (rule == 0) {
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = mxfp4_clamped(f[i], inv, 0);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = mxfp4_clamped(f[i], inv, 1);
  }
  uint32_t pk = e2m1_pair<0>(0u, f[0], f[1]);
  pk = e2m1_pair<1>(pk, f[2], f[3]);
  pk = e2m1_pair<2>(pk, f[4], f[5]);
  pk = e2m1_pair<3>(pk, f[6], f[7]);
  if (!live) return;
  packed[g] = pk;
  if (dq) {  // nibble * 2^k, exact in bf16 (two significant bits; sign of zero kept)
    const float s = pow2f(k);
    dq[g] = make_uint4(__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(pk, s, 0)),
                       __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(pk, s, 1)),
                       __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(pk, s, 2)),
                       __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(pk, s, 3)));
  }
  if ((g & 3) == 0) scale[g >> 2] = (uint8_t)(k + 127);
}

// As fp8_quant_wg (n_groups a multiple of 4).
template <int U, int NT>
DSV4_DEV void mxfp4_quant_wg(const uint4* __restrict__ x, int64_t wg, int64_t n_groups, int rule,
                             uint32_t* __restrict__ packed, uint8_t* __restrict__ scale, uint4* __restrict__ dq) {
  const int64_t g0 = wg * (U * NT) + threadIdx.x;
  uint4 v[U];
#pragma unroll
  for (int i = 0; i < U; ++i) v[i] = g0 + i * NT < n_groups ? x[g0 + i * NT] : make_uint4(0, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < U; ++i) mxfp4_quant_loaded(v[i], g0 + i * NT, g0 + i * NT < n_groups, rule, packed, scale, dq);
}

}  // namespace dsv4
