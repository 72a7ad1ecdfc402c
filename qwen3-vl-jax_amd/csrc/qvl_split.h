// fp32 values as two f16 terms of a power-of-two multiple (hi + lo), shared by the fp32 Dense (qvl_f32_split.hip)
// and the fp32 attention (qvl_f32_attn.hip) on the f16 matrix cores.
#pragma once
#include "qvl_kernels.h"

namespace qvl {

typedef _Float16 f16;
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// The power of two that takes values up to `mx` (finite, >= 0) into f16 range: mx * s in [2^14, 2^15).
// Clamped to normal fp32 values of s and 1 / s; zero and non-finite maxima give 1.
__device__ __forceinline__ float split_scale(float mx) {
  const int ex = (int)(__float_as_uint(mx) >> 23);   // biased exponent (mx >= 0); 0: zero or denormal
  if (ex == 0 || ex == 255) return mx > 0.f && ex == 0 ? 0x1p126f : 1.0f;
  return __uint_as_float((uint32_t)min(127 + 14 - (ex - 127), 253) << 23);
}

// hi + lo of one value. The empty asm pins the fp32 value: without it the compiler may form hi twice, once
// rounded straight from the product that gave t (v_fma_mixlo_f16) and once from t, and near a tie the two differ.
__device__ __forceinline__ void split1(float t, f16& hi, f16& lo) {
  asm("" : "+v"(t));
  hi = (f16)t;
  lo = (f16)(t - (float)hi);
}

__device__ __forceinline__ void split4(const f32x4& v, float s, f16x4& hi, f16x4& lo) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    f16 h, l;
    split1(v[e] * s, h, l);
    hi[e] = h;
    lo[e] = l;
  }
}

// Writes columns c..c+3 (c a multiple of 4) of a split row.
__device__ __forceinline__ void store_split4(f16* row, int c, const f16x4& hi, const f16x4& lo) {
  f16* g = row + (c >> 5) * 64 + (c & 31);
  *reinterpret_cast<f16x4*>(g) = hi;
  *reinterpret_cast<f16x4*>(g + 32) = lo;
}

}  // namespace qvl
