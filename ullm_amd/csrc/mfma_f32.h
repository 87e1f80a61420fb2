// Operands of v_mfma_f32_16x16x4_f32 in the order of a plain sum.  The instruction adds its four products one after the other,
// lane group 0's first, each sum rounded: with group g standing for k = 4 i + g in the i-th of four instructions, a chain of
// them over chunks of 16 gives the bits of fma(a[k], b[k], sum) for k = 0, 1, 2, ...
#pragma once
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

__device__ __forceinline__ float4 ld4_f32(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 ld4_f32(const bf16_t* p) {
  const uint2 u = *reinterpret_cast<const uint2*>(p);
  return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                     __uint_as_float(u.y & 0xffff0000u));
}

// Lane (r, g) brings values 4 g .. 4 g + 3 of row r's chunk of 16 and takes values g, 4 + g, 8 + g, 12 + g: a 4 x 4 transposition
// between registers and lane groups (four lane swaps inside the vector unit).
__device__ __forceinline__ f32x4_t in_order(const float4& v) {
#ifdef __HIP_DEVICE_COMPILE__
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v.x), __float_as_uint(v.z), false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v.y), __float_as_uint(v.w), false, false);
  const auto lo = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  return f32x4_t{__uint_as_float(lo[0]), __uint_as_float(lo[1]), __uint_as_float(hi[0]), __uint_as_float(hi[1])};
#else
  return f32x4_t{v.x, v.y, v.z, v.w};
#endif
}
