/*
 * gemm_split.h -- the workspace of the launches in which several workgroups
 * divide a tile's K (gemm_direct.hip, gemm_ring.hip, gemm_f32.hip): a ticket
 * per tile, zero between launches, then the partial sums. One per stream
 * serves all of them. Plain host arithmetic.
 */
#ifndef VX_AMD_GEMM_SPLIT_H
#define VX_AMD_GEMM_SPLIT_H

#include <cstdint>

namespace vxk {
namespace split {

constexpr int kMaxTiles = 1024;
constexpr int64_t kTicketBytes = kMaxTiles * 4;
/* The most that a stream keeps. By the time models below, over M, N up to
 * 16384 and K up to 262144, it costs a few large grids of K past 200000 up to
 * 14% (f32 9869 x 1212 x 248544 in 2 splits for 16, whose sums take 780 MiB);
 * half of it would cost up to 48%. */
constexpr int64_t kMaxBytes = (int64_t)128 << 20;

} // namespace split
} // namespace vxk

#endif /* VX_AMD_GEMM_SPLIT_H */
