// bf16_math.h - device helpers on bf16 pairs shared by the weight-path
// kernels (model_kernels.hip, gemm_tiles.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mckv {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float lo_f(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float hi_f(uint32_t u) { return __uint_as_float(u & 0xFFFF0000u); }
// Two fp32 -> bf16 round-to-nearest-even conversions in one v_cvt_pk_bf16_f32
// (a in the low half).
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){a, b}, bf16x2_t));
}
// SwiGLU of one gate / up pair.
__device__ __forceinline__ float silu_mul(float g, float u) {
    return g / (1.0f + expf(-g)) * u;
}

}  // namespace mckv
