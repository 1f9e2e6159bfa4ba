/*
 * vx_wave_ops.hip.h -- wave-wide reductions of the decoder's kernels
 * (decode.hip, prefill.hip), on VALU data movement.
 */
#ifndef VX_AMD_WAVE_OPS_HIP_H
#define VX_AMD_WAVE_OPS_HIP_H

#include <hip/hip_runtime.h>

namespace vxk {
namespace {

/* Wave-wide all-reduce with VALU data movement (DPP within 16-lane rows,
 * v_permlane16/32_swap across them) instead of LDS-crossbar shuffles. */
template <int kO> __device__ __forceinline__ float partner(float v) {
  static_assert(kO == 1 || kO == 2 || kO == 4 || kO == 8, "within a row");
  /* Lane i of a 16-lane row reads the lane differing in bit 3 (rotate by
   * 8), bit 2 (mirror within 8), bit 1 or bit 0 (quad permutes). */
  constexpr int ctrl = kO == 8 ? 0x128 : kO == 4 ? 0x141 : kO == 2 ? 0x4e : 0xb1;
  return __uint_as_float(
      __builtin_amdgcn_update_dpp(0u, __float_as_uint(v), ctrl, 0xf, 0xf, false));
}

/* Sum over groups of kN consecutive lanes (kN a power of two, <= 64); every
 * lane of a group ends with its group's sum. */
template <int kN> __device__ __forceinline__ float group_sum(float v) {
  if constexpr (kN >= 2) v += partner<1>(v);
  if constexpr (kN >= 4) v += partner<2>(v);
  if constexpr (kN >= 8) v += partner<4>(v);
  if constexpr (kN >= 16) v += partner<8>(v);
  if constexpr (kN >= 32) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v),
                                                    __float_as_uint(v), false,
                                                    false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  if constexpr (kN >= 64) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v),
                                                    __float_as_uint(v), false,
                                                    false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  return v;
}

__device__ __forceinline__ float wave_sum(float v) { return group_sum<64>(v); }

__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, partner<1>(v));
  v = fmaxf(v, partner<2>(v));
  v = fmaxf(v, partner<4>(v));
  v = fmaxf(v, partner<8>(v));
  {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v),
                                                    __float_as_uint(v), false,
                                                    false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v),
                                                    __float_as_uint(v), false,
                                                    false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  return v;
}

} // namespace
} // namespace vxk

#endif /* VX_AMD_WAVE_OPS_HIP_H */
