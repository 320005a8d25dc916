// q3h_math.h - scalar device math whose results are fixed to the bit by IEEE
// operations alone, so that the int8 path reproduces a CPU evaluation of the
// same formulas exactly.
#pragma once

#include <hip/hip_runtime.h>

namespace q3h {

// e^x: Cody & Waite (1980) argument reduction x = k ln2 + r, k = rint(x
// log2 e), ln 2 split in a 16-bit head and its tail; e^r by its Taylor series
// to r^7 (|r| <= 0.35: truncation < 6e-9 relative) in Horner form with fused
// multiply-adds; times 2^k built from the exponent bits. Error < 1 ulp
// measured; 0 below -86 (no subnormal results), +inf above 88.
__device__ __forceinline__ float exp_ieee(float x) {
  if (x != x) return x;
  if (x < -86.0f) return 0.0f;
  if (x > 88.0f) return __builtin_inff();
  const float k = rintf(__fmul_rn(x, 0x1.715476p+0f));
  float r = fmaf(k, -0x1.62e4p-1f, x);
  r = fmaf(k, -0x1.7f7d1cp-20f, r);
  float p = 0x1.a01a02p-13f;       // 1/7!
  p = fmaf(p, r, 0x1.6c16c2p-10f);  // 1/6!
  p = fmaf(p, r, 0x1.111112p-7f);   // 1/5!
  p = fmaf(p, r, 0x1.555556p-5f);   // 1/4!
  p = fmaf(p, r, 0x1.555556p-3f);   // 1/3!
  p = fmaf(p, r, 0.5f);
  p = fmaf(p, r, 1.0f);
  p = fmaf(p, r, 1.0f);
  const float scale = __builtin_bit_cast(float, (unsigned)((int)k + 127) << 23);
  return __fmul_rn(p, scale);
}

// SiLU(g) * u = g / (1 + e^-g) * u, each operation rounded once
__device__ __forceinline__ float silu_mul_ieee(float g, float u) {
  return __fmul_rn(__fdiv_rn(g, __fadd_rn(1.0f, exp_ieee(-g))), u);
}

// SiLU of the text projection: 0 below -80 (where e^-v would overflow)
__device__ __forceinline__ float silu_clamp_f(float v) {
  return v < -80.0f ? 0.0f : v / (1.0f + expf(-v));
}

// sinf, kept out of line
__host__ __device__ __attribute__((noinline)) inline float sin_far(float x) { return sinf(x); }

// sin(x)^2, the SnakeBeta term: of period pi and even, so x is reduced by the
// nearest multiple of pi and the sign of the result does not matter. pi is the
// sum of three floats: the first product is exact below 4e5 (k < 2^17; x and k
// p1 are multiples of 2^-23 and their difference is below 2), the second is
// rounded once in the result's own last place, and the third's (k 3.4e-15, which
// two floats left out) keeps that so where x is next to a multiple of pi. sin r,
// |r| <= pi / 2, by its Taylor series to r^13 (truncation < 7e-10) in Horner
// form. sin x within 3 units of 2^-24, relative (two roundings of r, one of the
// last step); beyond 4e5 by sinf. 17 instructions without a branch taken, where
// sinf's general reduction, inlined per output, made a decoder epilogue of 32
// values 9000 lines long.
__host__ __device__ __forceinline__ float sin_squared(float x) {
  float s;
  if (fabsf(x) < 4e5f) {
    const float k = rintf(x * 0x1.45f306p-2f);
    float r = fmaf(-k, 0x1.921fb6p+1f, x);
    r = fmaf(k, 0x1.777a5cp-24f, r);
    r = fmaf(k, 0x1.ee59dap-49f, r);
    const float r2 = r * r;
    float p = 0x1.612462p-33f;       // 1/13!
    p = fmaf(p, r2, -0x1.ae6456p-26f);  // -1/11!
    p = fmaf(p, r2, 0x1.71de3ap-19f);   // 1/9!
    p = fmaf(p, r2, -0x1.a01a02p-13f);  // -1/7!
    p = fmaf(p, r2, 0x1.111112p-7f);    // 1/5!
    p = fmaf(p, r2, -0x1.555556p-3f);   // -1/3!
    s = fmaf(r * r2, p, r);
  } else {
    s = sin_far(x);
  }
  return s * s;
}

// RoPE of the pair (a, b) = (x_i, x_{i + d/2}): a' = a c - b s, b' = b c + a s,
// the second product fused into the subtraction / addition
__device__ __forceinline__ void rope_pair(float &a, float &b, float c, float s) {
  const float a0 = a, b0 = b;
  a = fmaf(a0, c, -__fmul_rn(b0, s));
  b = fmaf(b0, c, __fmul_rn(a0, s));
}

// x = hi + mid + lo exactly, each a bf16 (returned as its 16 bits in the low
// half): hi the top 8 significant bits of x, mid the next 8, lo the last 8
// (an f32 significand has 24; each difference is exact in f32). For products
// whose other operand is exact in bf16 (all three part products are summed);
// where part products are dropped, the parts are rounded: split3_rn.
__device__ __forceinline__ void split3(float x, uint32_t &h, uint32_t &m, uint32_t &l) {
  const uint32_t u = __float_as_uint(x);
  const uint32_t hb = u & 0xffff0000u;
  const float r1 = x - __uint_as_float(hb);
  const uint32_t mb = __float_as_uint(r1) & 0xffff0000u;
  const float r2 = r1 - __uint_as_float(mb);
  h = hb >> 16;
  m = mb >> 16;
  l = __float_as_uint(r2) >> 16;
}

// The same for a (low halves) and b (high halves), hi and mid rounded to
// nearest: |mid| <= 2^-9 and |lo| <= 2^-18 of the binade's top, of either sign,
// so the part products below hi lo that a six-part product leaves out (mid lo,
// lo mid, lo lo) weigh at most 2^-24 of it and cancel on average. Cut off
// instead of rounded (split3) they reach 2^-21 and all have the product's sign:
// a result of two one-term products 9.2e-8 off (RMS) instead of 3.6e-8. As many
// instructions (the pair conversion of gfx950 packs as it rounds) and one more
// per value: hi of a value within half a bf16 step of the largest float would
// be infinite, so it is taken of the value limited to the largest bf16. (Parts
// below the smallest normal number, of values under 2^-102, may be lost.)
__device__ __forceinline__ void split3_rn(float a, float b, uint32_t &h, uint32_t &m,
                                          uint32_t &l) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  auto pack = [](float x, float y) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{x, y}), b2));
  };
  constexpr float kMax = 0x1.fep127f;
  h = pack(__builtin_amdgcn_fmed3f(a, -kMax, kMax), __builtin_amdgcn_fmed3f(b, -kMax, kMax));
  const float a1 = a - __uint_as_float(h << 16), b1 = b - __uint_as_float(h & 0xffff0000u);
  m = pack(a1, b1);
  l = pack(a1 - __uint_as_float(m << 16), b1 - __uint_as_float(m & 0xffff0000u));
}

}  // namespace q3h
