/*
 * flash_rows.h -- how the attention of few queries (flash_rows.hip) is
 * divided. Plain host arithmetic.
 */
#ifndef VX_AMD_FLASH_ROWS_H
#define VX_AMD_FLASH_ROWS_H

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

namespace vxk {
namespace rows {

/* A split launch's workspace: a ticket per item, zero between launches, then
 * the partial results. */
constexpr int kMaxSplitItems = 4096;
constexpr int64_t kTicketBytes = kMaxSplitItems * 4;

struct Plan {
  int mt;     /* 16-row tiles per item: 1 or 2 */
  int tiles;  /* items per (batch, KV head) */
  int splits; /* workgroups that divide an item's keys */
  int64_t ws_bytes;
};

struct Args {
  const uint16_t *q, *k, *v;
  uint16_t *o;
  float *lse;
  int64_t kv_total; /* batch * kv_heads */
  int rows;         /* queries per KV head: group * seq_q */
  int seq_q, seq_k;
  float scale_log2;
  bool causal;
};

} // namespace rows

void flash_rows_launch(const rows::Args &a, const rows::Plan &plan, int head_dim, char *ws,
                       hipStream_t stream);

} // namespace vxk

#endif /* VX_AMD_FLASH_ROWS_H */
