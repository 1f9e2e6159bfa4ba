/*
 * gemm_direct.h -- which shapes the register GEMM (gemm_direct.hip) takes,
 * and how it divides them. Plain host arithmetic.
 */
#ifndef VX_AMD_GEMM_DIRECT_H
#define VX_AMD_GEMM_DIRECT_H

#include "gemm_split.h"

#include <algorithm>
#include <cstdint>

namespace vxk {
namespace direct {

struct Plan {
  int mt;           /* 16-row blocks per wave: 1, 2 or 4 */
  bool along_k;     /* the waves of a workgroup share a tile and divide k */
  int tiles_m, tiles_n;
  int splits;       /* workgroups that divide a tile's k */
  int64_t ws_bytes; /* 0 without splits */
};

/* Eight columns at least (a lane's load); byte offsets of a tile's 64 rows of
 * A and 32 of B in 31 bits; a grid in 31 bits. */
inline bool shape_ok(int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb, int64_t ldc) {
  return m >= 1 && n >= 8 && k >= 1 && k <= (1 << 30) && lda >= k && ldb >= n && ldc >= n &&
         lda <= (1 << 23) && ldb <= (1 << 23) &&
         ((m + 15) / 16) * ((n + 127) / 128) <= (1 << 24);
}

/* Microseconds, from times on a 256-CU MI355X (4 to 8192 rows, K 64 to 12000,
 * within a third of the measured; 8 to 400000 rows and columns, K 1 to 127): a
 * launch takes 3, and a wave one block of 32 k in `block`; an A off the 4-byte
 * grid is loaded in words. Two operands of 4000^3, for instance: 128 blocks on
 * two rounds of 256-row tiles 215, with odd rows 340. */
inline double block_us(int mt, bool along_k, bool odd) {
  if (!along_k) {
    return odd ? 1.3 : 0.77;
  }
  return mt == 1 ? (odd ? 1.1 : 0.48) : mt == 2 ? (odd ? 1.1 : 0.75) : odd ? 1.6 : 0.95;
}

/* The division of least time by that model. `odd`: A off the 4-byte grid;
 * `cus` compute units; `may_split`: whether a workspace may be had. `us`
 * receives the time. Examples of what it weighs (bf16 -> f32, K = 4096): 8 x
 * 4096 in 8 splits 8.0 us, in 1 15.6, in 16 11.9; 512 x 4096 in 64-row tiles
 * 33, in 32-row tiles 43; 500 x 501 x 5001 in 32-row tiles and 4 splits 16.6,
 * in 16-row tiles and 2 25.1. */
inline Plan plan(int64_t m, int64_t n, int64_t k, bool odd, int cus, bool may_split, double *us) {
  Plan best{};
  *us = 1e30;
  const double blocks = (double)((k + 31) / 32);
  const int tiles_n = (int)((n + 127) / 128);
  auto consider = [&](int mt, bool along_k, int rows, int64_t splits) {
    const int64_t tiles_m = (m + rows - 1) / rows, tiles = tiles_m * tiles_n;
    const int64_t rounds = (tiles * splits + cus - 1) / cus;
    double t = 3.0 + (double)rounds * (along_k ? 0.5 + 0.5 * mt + blocks / (double)(4 * splits) * block_us(mt, true, odd)
                                               : 9.0 + blocks * block_us(mt, false, odd));
    if (along_k && mt == 4) {
      /* one to a CU: nothing covers a round's start and store (146800 x 40 x 16
       * in 9 rounds of these 46.8, in 3 of 256 rows 19.2); on two rounds the
       * time above is close (124 x 22574 x 648 27.4, in 32-row tiles 33.5) */
      t += 2.0 * (double)std::max<int64_t>(rounds - 2, 0);
    }
    if (splits > 1) {
      t += 1.0 + 0.6 * mt + 0.05 * (double)(splits * mt); /* the ticket, the other splits' sums */
    }
    if (t < *us) {
      *us = t;
      best.mt = mt;
      best.along_k = along_k;
      best.tiles_m = (int)tiles_m;
      best.tiles_n = tiles_n;
      best.splits = (int)splits;
      best.ws_bytes = splits > 1 ? split::kTicketBytes + tiles * splits * (int64_t)(mt * 16 * 128 * 4) : 0;
    }
  };
  consider(4, false, 256, 1);
  for (int mt = 4; mt >= 1; mt /= 2) {
    if (mt > 1 && m <= 8 * mt) {
      continue; /* half of the tile or more would be past the last row */
    }
    consider(mt, true, 16 * mt, 1);
    const int64_t tiles = (m + 16 * mt - 1) / (16 * mt) * tiles_n;
    /* one workgroup per CU, of at least 4 blocks of k a wave */
    const int64_t splits = std::min<int64_t>(cus / tiles, k / 512);
    if (may_split && splits > 1 && tiles <= split::kMaxTiles) {
      consider(mt, true, 16 * mt, splits);
    }
  }
  return best;
}

} // namespace direct
} // namespace vxk

#endif /* VX_AMD_GEMM_DIRECT_H */
