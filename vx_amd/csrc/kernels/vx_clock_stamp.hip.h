/*
 * vx_clock_stamp.hip.h -- the clock stamp that a caller may ask of a GEMM
 * launch (GemmArgs::stamp): workgroup 0 records the shader-clock counter and
 * the constant 100 MHz real-time counter at its start and end, so that the
 * clock the kernel ran at can be read. Null in ordinary launches; the branch
 * is uniform.
 */
#ifndef VX_AMD_CLOCK_STAMP_HIP_H
#define VX_AMD_CLOCK_STAMP_HIP_H

#include <hip/hip_runtime.h>

#include <cstdint>

namespace vxk {
namespace {

struct ClockStamp {
  uint64_t *to;
  uint64_t clk = 0, rt = 0;

  __device__ __forceinline__ explicit ClockStamp(uint64_t *stamp)
      : to(blockIdx.x == 0 ? stamp : nullptr) {
    if (to) {
      clk = __builtin_amdgcn_s_memtime();
      rt = __builtin_amdgcn_s_memrealtime();
    }
  }
  /* Before each return of workgroup 0's first thread. */
  __device__ __forceinline__ void end() const {
    if (to && threadIdx.x == 0) {
      const uint64_t clk1 = __builtin_amdgcn_s_memtime();
      const uint64_t rt1 = __builtin_amdgcn_s_memrealtime();
      to[0] = clk;
      to[1] = rt;
      to[2] = clk1;
      to[3] = rt1;
    }
  }
};

} // namespace
} // namespace vxk

#endif /* VX_AMD_CLOCK_STAMP_HIP_H */
