/*
 * vx_mfma16.hip.h -- v_mfma_f32_16x16x32 on bf16 or f16 operands held as
 * four words (eight values of k a lane).
 */
#ifndef VX_AMD_MFMA16_HIP_H
#define VX_AMD_MFMA16_HIP_H

#include <hip/hip_runtime.h>

#include <cstdint>

namespace vxk {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <bool kBf16>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (kBf16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
        __builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
        0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(
        __builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
        0);
  }
}

} // namespace
} // namespace vxk

#endif /* VX_AMD_MFMA16_HIP_H */
