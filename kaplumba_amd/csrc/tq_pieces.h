// Exact products of f32 operands on v_mfma_f32_16x16x32_bf16: operands as bf16
// pieces that sum to them (tq_rotate.hip, tq_append_few.hip).
#pragma once

#include "tq_common.h"

namespace tq {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t mfma_bf16(u32x4_t a, u32x4_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0,
                                                 0, 0);
}

// Eight f32 values as NP bf16 pieces each (round to nearest even, exact remainders).
template <int NP>
__device__ __forceinline__ void split8(const float (&v)[8], u32x4_t (&w)[NP]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float a = v[2 * j], b = v[2 * j + 1];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const bf16x2_t x = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
      const uint32_t u = __builtin_bit_cast(uint32_t, x);
      w[p][j] = u;
      a = __fsub_rn(a, __uint_as_float(u << 16));
      b = __fsub_rn(b, __uint_as_float(u & 0xffff0000u));
    }
  }
}

}  // namespace tq
