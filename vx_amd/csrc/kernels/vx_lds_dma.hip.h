/*
 * vx_lds_dma.hip.h -- buffer-to-LDS loads and the waits that order them.
 */
#ifndef VX_AMD_LDS_DMA_HIP_H
#define VX_AMD_LDS_DMA_HIP_H

#include <hip/hip_runtime.h>

#include <cstdint>

namespace vxk {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
#define VX_LDS __attribute__((address_space(3)))

/* Wait until at most `n` of this wave's vector memory operations are
 * outstanding (vmcnt n; lgkmcnt and expcnt untouched). */
template <int n>
__device__ __forceinline__ void wait_vm() {
  static_assert(n >= 0 && n < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8));
}

/* Wait until at most `newer` (0..kMax) whole stages of this wave's loads are
 * outstanding; each stage is kPer loads. */
template <int kMax, int kPer>
__device__ __forceinline__ void wait_stages(int newer) {
  if constexpr (kMax == 0) {
    wait_vm<0>();
  } else if (newer >= kMax) {
    wait_vm<kMax * kPer>();
  } else {
    wait_stages<kMax - 1, kPer>(newer);
  }
}

/* One 16-byte-per-lane load from the buffer `rsrc` at byte offset `voff`
 * into LDS at `lds` + 16*lane. Written as assembly so the compiler neither
 * waits for it at every LDS read (it cannot tell which ring slot the load
 * fills) nor drops the barrier-time vmcnt(0) it adds for a fenced barrier:
 * the kernel orders these loads itself with wait_vm and lds_barrier. The
 * nop covers the one wait state between the M0 write and its use. */
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm" /* m0 is reserved: declared */
__device__ __forceinline__ void dma16(i32x4 rsrc, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
               :
               : "v"(voff), "s"(rsrc), "s"(lds)
               : "memory", "m0");
}
#pragma clang diagnostic pop

/* Workgroup barrier without the release fence __syncthreads carries (that
 * fence waits for every outstanding global load, the prefetches included).
 * LDS reads are drained first so a slot is never refilled under a reader. */
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xc07f); /* lgkmcnt(0) */
  asm volatile("s_barrier" ::: "memory");
}

/* Raw 32-bit-dword buffer of `bytes` bytes at `base`: a load past its end
 * returns zeros. */
__device__ __forceinline__ i32x4 buffer_rsrc(const void *base, int bytes) {
  const uint64_t a = (uint64_t)base;
  i32x4 r;
  r[0] = (int)(uint32_t)a;
  r[1] = (int)((uint32_t)(a >> 32) & 0xffffu); /* stride 0 */
  r[2] = bytes;
  r[3] = 0x00020000;
  return r;
}

} // namespace
} // namespace vxk

#endif /* VX_AMD_LDS_DMA_HIP_H */
