/*
 * gemm_f32.h -- which kernel of the f32 MFMA GEMM (gemm_f32.hip) takes a shape,
 * and the choice of its splits. Plain host arithmetic.
 */
#ifndef VX_AMD_GEMM_F32_H
#define VX_AMD_GEMM_F32_H

#include "gemm_split.h"

namespace vxk {
namespace f32 {

constexpr int kTile = 128;
constexpr int kPart = kTile * kTile * 4; /* bytes of a split's sums of a tile */
/* K from which the bf16 planes are taken: below it a tile is its loads, its
 * start and writing C, and f32 MFMAs do with a sixth of the LDS (planes and
 * f32: 4096^2 x 96 39.7 us and 36.0, x 128 44.1 and 43.6, x 160 49.3 and 51.7;
 * 3000^2 x 128 32.3 and 33.7; 2^20 x 8 x 128 314 and 290, x 192 411 and 421). */
constexpr int64_t kPlanesMinK = 128;

inline int64_t tiles(int64_t m, int64_t n) {
  return ((m + kTile - 1) / kTile) * ((n + kTile - 1) / kTile);
}
inline int64_t ws_bytes(int64_t m, int64_t n, int splits) {
  return split::kTicketBytes + tiles(m, n) * splits * (int64_t)kPart;
}

/* Splits of least time on a 256-CU MI355X (one workgroup to a CU): 1.15 us a
 * stage of K, 4 a round, and for a split its sums' way to memory and back. */
inline int splits(int64_t m, int64_t n, int64_t k, int cus, bool may_split) {
  const int64_t t = tiles(m, n), stages = (k + 31) / 32;
  if (!may_split || t > split::kMaxTiles) {
    return 1;
  }
  int best = 1;
  double least = 1e30;
  for (int s = 1; s <= 16 && (s == 1 || (stages / s >= 4 && ws_bytes(m, n, s) <= split::kMaxBytes));
       ++s) {
    const double rounds = (double)((t * s + cus - 1) / cus);
    double us = rounds * (4.0 + 1.15 * (double)stages / s);
    if (s > 1) {
      us += 3.0 + (double)(t * s) * kPart * 2 / 5e6;
    }
    if (us < least) {
      least = us;
      best = s;
    }
  }
  return best;
}

} // namespace f32

} // namespace vxk

#endif /* VX_AMD_GEMM_F32_H */
