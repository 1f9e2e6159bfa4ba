/*
 * gemm_ring.h -- the choice of tile and splits of the 128x128- and 256x128-tile
 * GEMM (gemm_ring.hip). Plain host arithmetic.
 */
#ifndef VX_AMD_GEMM_RING_H
#define VX_AMD_GEMM_RING_H

#include "gemm_split.h"

#include <algorithm>

namespace vxk {
namespace ring {

constexpr int kTile = 128;

inline int64_t tiles(int64_t m, int64_t n) {
  return ((m + kTile - 1) / kTile) * ((n + kTile - 1) / kTile);
}
inline int64_t ws_bytes(int64_t m, int64_t n, int splits) {
  return split::kTicketBytes + tiles(m, n) * splits * (int64_t)(kTile * kTile * 4);
}

/* Microseconds on a 256-CU MI355X: a stage of K takes 0.53 where CUs have two
 * workgroups and 0.34 where they have one, a round of two per CU 2.5 to start
 * and store, and a split its sums' way to memory and back. */
inline double us(int64_t m, int64_t n, int64_t k, int splits, int cus) {
  const int64_t units = tiles(m, n) * splits, slots = 2 * (int64_t)cus;
  const int64_t full = units / slots, rest = units % slots;
  const double stages = (double)(k / 32) / splits;
  double t = 3.0 + 2.5 * (double)(full + (rest > 0));
  t += stages * (0.53 * (double)full + (rest > cus ? 0.53 : rest > 0 ? 0.34 : 0.0));
  if (splits > 1) {
    t += 3.0 + (double)units * kTile * kTile * 8 / 5e6;
  }
  return t;
}

/* Whether an undivided launch takes tiles of 256x128, one workgroup to a CU:
 * where CUs would have two of 128x128 and these fit one to each. They read B
 * half as often, which counts when it comes from HBM. New inputs each pass,
 * bf16: 512 x 11008 x 4096 91 -> 79 us (the same ones again 70 -> 66), 1024 x
 * 5120 x 4096 91 -> 75, 300 x 12288 x 4096 85 -> 70, 512 x 11008 x 2048 50 ->
 * 44 (the same ones 36 -> 37). Shorter K keeps the smaller tiles: x 1024 30 ->
 * 28 (22 -> 23), x 256 13.7 -> 14.4. */
inline bool tall(int64_t m, int64_t n, int64_t k, int cus) {
  return tiles(m, n) > cus && (m + 2 * kTile - 1) / (2 * kTile) * ((n + kTile - 1) / kTile) <= cus &&
         k >= 2048;
}

/* Splits of least time by that model. */
inline int splits(int64_t m, int64_t n, int64_t k, int cus, bool may_split) {
  int best = 1;
  if (may_split && tiles(m, n) <= split::kMaxTiles) {
    for (int s = 2; s <= 8 && k / 32 / s >= 8 && ws_bytes(m, n, s) <= split::kMaxBytes; ++s) {
      if (us(m, n, k, s, cus) < us(m, n, k, best, cus)) {
        best = s;
      }
    }
  }
  return best;
}

} // namespace ring

} // namespace vxk

#endif /* VX_AMD_GEMM_RING_H */
