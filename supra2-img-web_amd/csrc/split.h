// float32 operands as three bfloat16 terms, for products on the bf16 matrix cores of gfx950.
#pragma once

#include "common.h"

namespace sa {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// x = h + m + l with h, m, l the bfloat16 roundings of x, x - h and x - h - m (both differences exact):
// the three terms hold all 24 bits of x. 11 VALU instructions per pair of values.
struct Split8 {
  u32x4 h, m, l;  // 8 bfloat16 each, in order
};

__device__ __forceinline__ uint32_t cvt_pk_bf16(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

__device__ __forceinline__ void split_pair(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = cvt_pk_bf16(a, b);
  const float ra = a - __uint_as_float(h << 16), rb = b - __uint_as_float(h & 0xffff0000u);
  m = cvt_pk_bf16(ra, rb);
  const float sa = ra - __uint_as_float(m << 16), sb = rb - __uint_as_float(m & 0xffff0000u);
  l = cvt_pk_bf16(sa, sb);
}

__device__ __forceinline__ Split8 split8(f32x4 a, f32x4 b) {
  Split8 s;
  uint32_t h, m, l;
  split_pair(a[0], a[1], h, m, l);
  s.h[0] = h, s.m[0] = m, s.l[0] = l;
  split_pair(a[2], a[3], h, m, l);
  s.h[1] = h, s.m[1] = m, s.l[1] = l;
  split_pair(b[0], b[1], h, m, l);
  s.h[2] = h, s.m[2] = m, s.l[2] = l;
  split_pair(b[2], b[3], h, m, l);
  s.h[3] = h, s.m[3] = m, s.l[3] = l;
  return s;
}

__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

}  // namespace sa
