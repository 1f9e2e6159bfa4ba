/*
 * vx_clock_stamp.hip.h -- the clock stamp that a caller may ask of a GEMM
 * launch (GemmArgs::stamp): workgroup 0 records the shader-clock counter and
 * the constant 100 MHz real-time counter at its start and end, so that the
 * clock the kernel ran at can be read. Ordinary launches are kernels built
 * without it: the branch on a null pointer was 0.1 us of the smallest calls and
 * 0.4 of 77 us at 512 x 11008 x 4096.
 */
#ifndef VX_AMD_CLOCK_STAMP_HIP_H
#define VX_AMD_CLOCK_STAMP_HIP_H

#include <hip/hip_runtime.h>

#include <cstdint>

namespace vxk {
namespace {

template <bool kOn> struct ClockStamp {
  uint64_t *to; /* workgroup 0's, or null */

  __device__ __forceinline__ explicit ClockStamp(uint64_t *stamp)
      : to(blockIdx.x == 0 ? stamp : nullptr) {
    put(0);
  }
  /* Before each return of workgroup 0's first thread. */
  __device__ __forceinline__ void end() const { put(2); }

private:
  __device__ __forceinline__ void put(int at) const {
    if (to && threadIdx.x == 0) {
      to[at] = __builtin_amdgcn_s_memtime();
      to[at + 1] = __builtin_amdgcn_s_memrealtime();
    }
  }
};

template <> struct ClockStamp<false> {
  __device__ __forceinline__ explicit ClockStamp(uint64_t *) {}
  __device__ __forceinline__ void end() const {}
};

} // namespace
} // namespace vxk

#endif /* VX_AMD_CLOCK_STAMP_HIP_H */
