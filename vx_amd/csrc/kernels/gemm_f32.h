/*
 * gemm_f32.h -- launcher of the f32 MFMA GEMM (gemm_f32.hip).
 */
#ifndef VX_AMD_GEMM_F32_H
#define VX_AMD_GEMM_F32_H

#include "../vx_kernels.h"

namespace vxk {
namespace f32 {
constexpr int kTile = 128;
}
void gemm_f32_launch(const GemmArgs &g, hipStream_t s);
} // namespace vxk

#endif /* VX_AMD_GEMM_F32_H */
