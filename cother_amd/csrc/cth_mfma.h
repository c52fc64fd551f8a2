// cth_mfma.h: operands and products of the reduced-precision contraction on
// the matrix cores (precision 1: BF16, 2: FP16).
//
// v_mfma_f32_32x32x16 (lane l, 64 lanes): A holds row l%32, k = 8*(l/32) +
// 0..7; B holds column l%32, the same k; the 16 accumulators of lane l hold
// column l%32, rows 8*(r/4) + 4*(l/32) + r%4 for r = 0..15 (checked on the
// device by cth_selftest_mfma).
#pragma once
#include <hip/hip_runtime.h>

typedef short v8s __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

// round to nearest even (the operands are finite and >= 0)
template <int kPrec>
__device__ __forceinline__ uint16_t mfma_operand(float x) {
  if constexpr (kPrec == 1) {
    uint32_t u = __float_as_uint(x);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
  } else {
    return __builtin_bit_cast(uint16_t, (_Float16)x);
  }
}

template <int kPrec>
__device__ __forceinline__ v16f mfma(v8s a, v8s b, v16f acc) {
  if constexpr (kPrec == 1)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), acc, 0,
                                                   0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), acc, 0, 0,
                                                  0);
}
