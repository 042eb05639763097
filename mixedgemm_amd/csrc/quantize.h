// The arithmetic of the quantizers, shared by the kernels that store codes to memory and the one that keeps them in LDS.
#pragma once
#include "mg_common.h"

namespace mg {

// E8M0 byte of the block scale from the bits of amax (a non-negative float).
// MAX = fm * 2^pm with fm in [0.5,1): the exponent steps up by one when the
// mantissa of amax exceeds the mantissa of MAX, which the add below carries
// into the exponent field.  `fmt` may differ between the lanes of a wave.
__device__ __forceinline__ int scale_byte(float amax, int fmt) {
  const unsigned thr = fmt == kFmtE2M1 ? 0x400000u : 0x600000u;  // 6 = 1.5*4, 28 = 1.75*16, 448 = 1.75*256
  const int pm = fmt == kFmtE2M1 ? 3 : (fmt == kFmtE3M2 ? 5 : 9);
  const unsigned bits = __float_as_uint(amax);
  int byte = (int)((bits + (0x7FFFFFu - thr)) >> 23) + 1 - pm;
  byte = byte < 0 ? 0 : byte;
  return amax == 0.0f ? 126 : byte;
}

// roundf(x * rs) for a bf16 value x and a power of two rs, as one multiplication and one round-to-nearest-even:
// rs1 = rs * (1 + 2^-12).  x * rs has at most 8 significant bits, so x * rs1 is exact in fp32 (21 bits), a
// tie n + 0.5 moves off the tie away from zero, and every other value stays on its side of the nearest tie
// (it is at least one 8-bit step from it, the nudge is 2^-12 of the value).  The sign of zero is kept.
__device__ __forceinline__ float round_scaled(float x, float rs1) { return __builtin_rintf(x * rs1); }

// Sum of a double over the 64 lanes of a wave, the same value in every lane: four data-parallel-primitive steps inside
// the rows of 16 lanes (two register moves and an add each, no trip through the LDS crossbar), then the four row sums
// through scalar registers.
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(uint32_t)b, CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), CTRL, 0xF, 0xF, true);
  return v + __builtin_bit_cast(double, ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}
__device__ __forceinline__ double wave_sum(double v) {
  v = dpp_add<0xB1>(v);    // quad_perm [1, 0, 3, 2]
  v = dpp_add<0x4E>(v);    // quad_perm [2, 3, 0, 1]
  v = dpp_add<0x141>(v);   // row_half_mirror: the other quad of the 8
  v = dpp_add<0x140>(v);   // row_mirror: the other 8 of the 16
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  double rows[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)b, 16 * r), hi = __builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), 16 * r);
    rows[r] = __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
  }
  return (rows[0] + rows[1]) + (rows[2] + rows[3]);
}

// Half a block (16 gathered values, lane pair 2b / 2b + 1 holds block b): the pair's absmax by one cross-lane
// step, the scale byte, the codes; `half` (0 or 1) says which 16 elements these are.  `sink` takes the scale byte (first
// lane of a pair) and the 16 codes: 8 bytes of E2M1, 12 of E3M2 or 16 of E4M3.
template <class Sink>
__device__ __forceinline__ void quantize_half(const float (&f)[16], int fmt, int half, Sink sink) {
  float amax = 0.0f;
#pragma unroll
  for (int p = 0; p < 16; p += 2) amax = __builtin_fmaxf(__builtin_fmaxf(amax, __builtin_fabsf(f[p])), __builtin_fabsf(f[p + 1]));
  // quad_perm [1, 0, 3, 2]: the other lane of the pair
  const float other = __uint_as_float((unsigned)__builtin_amdgcn_mov_dpp((int)__float_as_uint(amax), 0xB1, 0xF, 0xF, true));
  amax = __builtin_fmaxf(amax, other);
  const int byte = scale_byte(amax, fmt);
  const float rs1 = __uint_as_float(((unsigned)(254 - byte) << 23) | 0x800u);
  float v[16];
#pragma unroll
  for (int p = 0; p < 16; ++p) v[p] = round_scaled(f[p], rs1);
  if (half == 0) sink.scale(byte);
  if (fmt == kFmtE2M1) {
    v2u out;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      unsigned w = 0;
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[8 * j + 0], v[8 * j + 1], 1.0f, 0);
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[8 * j + 2], v[8 * j + 3], 1.0f, 1);
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[8 * j + 4], v[8 * j + 5], 1.0f, 2);
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[8 * j + 6], v[8 * j + 7], 1.0f, 3);
      out[j] = w;
    }
    sink.codes(out);
  } else {
    if (fmt == kFmtE3M2) {
      // 16 codes are the first 96 bits of the 32-code conversion
      v32bf h;
#pragma unroll
      for (int p = 0; p < 16; ++p) h[p] = (__bf16)v[p];
#pragma unroll
      for (int p = 16; p < 32; ++p) h[p] = (__bf16)0.0f;
      const v6u w = __builtin_amdgcn_cvt_scalef32_pk32_bf6_bf16(h, 1.0f);
      sink.codes(v3u{w[0], w[1], w[2]});
    } else {
      unsigned out[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const v2bf lo = {(__bf16)v[4 * j + 0], (__bf16)v[4 * j + 1]};
        const v2bf hi = {(__bf16)v[4 * j + 2], (__bf16)v[4 * j + 3]};
        v2s z = {0, 0};
        z = __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(z, lo, 1.0f, false);
        z = __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(z, hi, 1.0f, true);
        out[j] = __builtin_bit_cast(unsigned, z);
      }
      sink.codes(v4u{out[0], out[1], out[2], out[3]});
    }
  }
}

// The scale of RMSNorm for a row whose squares sum to `sum` (accumulated in fp64), in the arithmetic of the usual fp32
// implementation: var = fl32(sum / K), r = fl32(1 / sqrt(fl32(var + eps))).  Between the roundings to fp32 neither is an fp64 division or
// square root, but the quotient is a product with inv_k = 1.0 / K corrected once by its exact residual (the correctly rounded one in
// each of 40000 random cases), and the root the hardware's estimate of 2^-23 with one third-order step (0.97 units in the last place
// of a double at most in as many; a square root followed by a division: 1.42).  The rounding to fp32 hides the difference but for one
// value in 2^28.  15 instructions instead of the compiler's ~90.  Infinite and NaN sums, and a sum of zero with eps = 0, as by a
// division and a square root.
__device__ __forceinline__ float rms_scale(double sum, int K, double inv_k, float eps) {
  const double q = sum * inv_k, left = __builtin_fma(-q, (double)K, sum);
  const float var = (float)(left == left ? __builtin_fma(left, inv_k, q) : q);
  const double v = (double)(var + eps), y = __builtin_amdgcn_rsq(v);
  const double e = __builtin_fma(-(v * y), y, 1.0);
  return (float)(e == e ? __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y) : y);
}
// Two channels of y = bf16(gamma * bf16(x * r)), both products in fp32.
__device__ __forceinline__ unsigned rms_apply(unsigned x, unsigned gamma, float r) {
  const float h0 = (float)(__bf16)(__uint_as_float(x << 16) * r);
  const float h1 = (float)(__bf16)(__uint_as_float(x & 0xffff0000u) * r);
  const v2bf y = {(__bf16)(__uint_as_float(gamma << 16) * h0), (__bf16)(__uint_as_float(gamma & 0xffff0000u) * h1)};
  return __builtin_bit_cast(unsigned, y);
}
// The same on two gathered channels; x and the weights as floats that hold bf16 values.
__device__ __forceinline__ void rms_apply(float& x0, float& x1, unsigned gamma0, unsigned gamma1, float r) {
  const v2bf h = {(__bf16)(x0 * r), (__bf16)(x1 * r)};
  const unsigned hb = __builtin_bit_cast(unsigned, h);
  const v2bf y = {(__bf16)(__uint_as_float(gamma0) * __uint_as_float(hb << 16)),
                  (__bf16)(__uint_as_float(gamma1) * __uint_as_float(hb & 0xffff0000u))};
  const unsigned yb = __builtin_bit_cast(unsigned, y);
  x0 = __uint_as_float(yb << 16);
  x1 = __uint_as_float(yb & 0xffff0000u);
}

}  // namespace mg
