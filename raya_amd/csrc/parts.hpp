// fp32 values as sums of three bfloat16 parts, and the matrix instruction that multiplies
// parts (gemm_kernel.hpp has the arithmetic and its error).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace raya {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t uint32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t uint32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx16 mfma_bf16(bf16x8 a, bf16x8 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// The three bfloat16 parts of x (low half of each word) and y (high half): 11 VALU operations.
// (v_dot2_f32_bf16 would take x - x0 in one operation, but runs at half rate: no faster.)
__device__ __forceinline__ uint32_t to_bf16x2(float x, float y) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2{x, y}, bf16x2));
}
__device__ __forceinline__ void split3(float x, float y, uint32_t (&p)[3]) {
    p[0] = to_bf16x2(x, y);
    x -= __uint_as_float(p[0] << 16);
    y -= __uint_as_float(p[0] & 0xffff0000u);
    p[1] = to_bf16x2(x, y);
    x -= __uint_as_float(p[1] << 16);
    y -= __uint_as_float(p[1] & 0xffff0000u);
    p[2] = to_bf16x2(x, y);
}

}  // namespace raya
