// float32 operands as three bfloat16 terms, for products on the bf16 matrix cores of gfx950.
#pragma once

#include "common.h"

namespace sa {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// x = h + m + l with h, m, l the bfloat16 roundings of x, x - h and x - h - m (both differences exact):
// the three terms hold all 24 bits of x from 2^-110 up. Below that l, and then m, run out of exponent: they are
// short by up to 2^-134 (20 bits are left at 2^-114, 8 at 2^-126, none below 2^-134). So the kernels either split kUp
// x, a multiple of 2^-125 for every float32 (from 2^104 up it is infinite, which their checks of the sums
// see), or compare their sums with what such operands may have cost them, and fall back to fp32 products.
// 11 VALU instructions per pair of values, 13 with the scaling.
constexpr float kUp = 0x1p24f, kDown = 0x1p-24f;

struct Split8 {
  u32x4 h, m, l;  // 8 bfloat16 each, in order
};

__device__ __forceinline__ uint32_t cvt_pk_bf16(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

// The terms of scale * a and scale * b. EXACT: of the products before their rounding to float32 (for a scale that
// is no power of two); otherwise the products are rounded first, which an fma would not make more
// exact, but at twice the issue time of the subtraction.
template <bool EXACT>
__device__ __forceinline__ void split_pair(float a, float b, float scale, uint32_t& h, uint32_t& m, uint32_t& l) {
#pragma clang fp contract(off)
  const float xa = a * scale, xb = b * scale;
  h = cvt_pk_bf16(xa, xb);
  const float ha = __uint_as_float(h << 16), hb = __uint_as_float(h & 0xffff0000u);
  const float ra = EXACT ? fmaf(a, scale, -ha) : xa - ha, rb = EXACT ? fmaf(b, scale, -hb) : xb - hb;
  m = cvt_pk_bf16(ra, rb);
  const float sa = ra - __uint_as_float(m << 16), sb = rb - __uint_as_float(m & 0xffff0000u);
  l = cvt_pk_bf16(sa, sb);
}

template <bool EXACT = false>
__device__ __forceinline__ Split8 split8(f32x4 a, f32x4 b, float scale = 1.f) {
  Split8 s;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x4& v = i < 2 ? a : b;
    const int e = 2 * (i & 1);
    uint32_t h, m, l;
    split_pair<EXACT>(v[e], v[e + 1], scale, h, m, l);
    s.h[i] = h, s.m[i] = m, s.l[i] = l;
  }
  return s;
}

__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

}  // namespace sa
