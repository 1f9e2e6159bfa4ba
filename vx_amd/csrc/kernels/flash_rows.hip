/*
 * flash_rows.hip -- attention forward of few queries over a long cache
 * (decode, and short chunks), bf16 in, f32 accumulate, bf16 out, f32
 * log-sum-exp: the same results as flash_attn.hip up to rounding.
 *
 * What bounds it is reading K and V once, so an item is all queries of one
 * (batch, KV head), the group's heads together (their rows of Q and O lie
 * together), in tiles of 16 rows, one or two of them on one reading. The
 * four waves of a workgroup take every fourth block of 32 keys, and as many
 * workgroups divide an item's keys as fill the CUs.
 *
 * K and V go from memory into MFMA operands, two blocks ahead and without
 * LDS (v_mfma_f32_16x16x32_bf16):
 *   S^T[key][q] = K Q^T: lane (l16, g) loads 16 bytes of row l16 per 32 d.
 *   O^T[d][q] += V^T P^T: the accumulators of two S^T tiles hold the keys
 *     4 g + e and 16 + 4 g + e of query l16, which in that order are the 8
 *     k-slots of P^T's operand; the lane loads its kD / 16 columns of those
 *     8 rows of V, and v_perm turns that block into V^T's operands, one per
 *     column.
 * The waves meet in LDS, the splits in a workspace: each leaves its max, sum
 * and unnormalised output past the caches that other XCDs do not see and
 * takes a ticket; the one with the last ticket adds them up in order.
 *
 * Against flash_attn.hip's kernel with a head's 1 query in its 128 rows: 8
 * sequences, 32 heads on 4, one query over 4096 keys 60 -> 16.6 us (4.0 TB/s
 * of K and V); 16 sequences, 64 heads on 8, over 8192 keys 600 -> 93 us
 * (5.8 TB/s). Four 16-row tiles on one reading need every register there is
 * and spill: 4 x 32 heads on 4, 8 queries 34 us, with two tiles 17.4.
 */
#include "../vx_hip_common.h"
#include "flash_rows.h"
#include "vx_mfma16.hip.h"

#include <cmath>

namespace vxk {
namespace {

constexpr int kThreads = 256;
constexpr int kKeys = 32;      /* per block */
constexpr float kSlack = 8.0f; /* base-2 headroom of the stale row max */
constexpr uint32_t kOut = 0x80000000u; /* past every range: zeros */

struct KernelArgs {
  rows::Args a;
  int tiles, splits;
  char *ws;
};

/* Over the four lanes that share lane % 16. */
__device__ __forceinline__ float over_g_max(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}
__device__ __forceinline__ float over_g_sum(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const f32x2 v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

template <int kD, int kMT>
__global__ __launch_bounds__(kThreads, kMT == 1 ? 2 : 1) void flash_rows(KernelArgs p) {
  constexpr int kSteps = kD / 32;  /* MFMA steps over d of a score tile */
  constexpr int kCols = kD / 16;   /* d per lane of V: 8 or 4 */
  constexpr int kVW = kCols / 2;   /* words of them */
  constexpr int kRow = kD * 2;     /* bytes */
  constexpr int kPad = kD + 4;     /* floats between LDS rows */
  constexpr int kRows = 16 * kMT;
  const rows::Args &a = p.a;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15;
  const int g = lane >> 4;
  /* the tiles of one reading of K and V far apart in the launch order, on one
   * XCD where the number of readings is a multiple of 8 */
  const int readings = (int)a.kv_total * p.splits;
  const int tile = blockIdx.x / readings;
  const int split = blockIdx.x % readings % p.splits;
  const int64_t kv = blockIdx.x % readings / p.splits;
  const int item = (int)kv * p.tiles + tile;
  const int row0 = tile * kRows;

  const int nb = (a.seq_k + kKeys - 1) / kKeys;
  const int b1 = (int)((int64_t)nb * (split + 1) / p.splits);
  int blk = (int)((int64_t)nb * split / p.splits) + wave;
  const int bytes = a.seq_k * kRow;
  const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(a.k + kv * a.seq_k * kD), (short)0, bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(a.v + kv * a.seq_k * kD), (short)0, bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t qr = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(a.q + (kv * a.rows + row0) * kD), (short)0, min(a.rows - row0, kRows) * kRow,
      0x00020000);

  u32x4 qf[kMT][kSteps]; /* zeros past the last row */
#pragma unroll
  for (int t = 0; t < kMT; ++t) {
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      qf[t][s] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                               qr, (16 * t + l16) * kRow + 64 * s + 16 * g, 0, 0));
    }
  }
  /* The last key each of the lane's queries sees, and the least of them. */
  const int shift = a.seq_k - a.seq_q;
  int limit[kMT];
#pragma unroll
  for (int t = 0; t < kMT; ++t) {
    limit[t] = a.causal ? (row0 + 16 * t + l16) % a.seq_q + shift : a.seq_k - 1;
  }
  const int all_see = a.causal ? min(shift, a.seq_k - 1) : a.seq_k - 1;

  struct Keys {
    u32x4 f[2][kSteps];
  };
  struct Values {
    uint32_t f[8][kVW];
  };
  const uint32_t k_at = (uint32_t)(l16 * kRow + 16 * g);
  const uint32_t v_at = (uint32_t)(4 * g * kRow + l16 * (2 * kCols));
  /* Blocks from b1 on and keys past the last load zeros. */
  auto load_k = [&](Keys &d, int b) {
    const uint32_t at = b < b1 ? (uint32_t)(b * kKeys * kRow) : kOut;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
        d.f[h][s] = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                       kr, (int)(at + k_at + (uint32_t)(16 * h * kRow + 64 * s)), 0, 0));
      }
    }
  };
  auto load_v = [&](Values &d, int b) {
    const uint32_t at = b < b1 ? (uint32_t)(b * kKeys * kRow) : kOut;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int off = (int)(at + v_at + (uint32_t)((16 * (e >> 2) + (e & 3)) * kRow));
      if constexpr (kVW == 4) {
        const u32x4 w = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(vr, off, 0, 0));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          d.f[e][i] = w[i];
        }
      } else {
        const u32x2 w = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(vr, off, 0, 0));
        d.f[e][0] = w[0];
        d.f[e][1] = w[1];
      }
    }
  };

  f32x4 o[kMT][kCols];
  float m_run[kMT], l_run[kMT]; /* l: over this lane's keys */
#pragma unroll
  for (int t = 0; t < kMT; ++t) {
    m_run[t] = -INFINITY;
    l_run[t] = 0.0f;
#pragma unroll
    for (int j = 0; j < kCols; ++j) {
      o[t][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }

  auto step = [&](int b, Keys &kf, Values &vf) {
    f32x4 s[kMT][2];
#pragma unroll
    for (int d = 0; d < kSteps; ++d) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int t = 0; t < kMT; ++t) {
          s[t][h] = mfma16<true>(kf.f[h][d], qf[t][d],
                                 d == 0 ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : s[t][h]);
        }
      }
    }
    load_k(kf, b + 8);
    const bool mask = (b + 1) * kKeys - 1 > all_see;
    u32x4 pt[kMT];
#pragma unroll
    for (int t = 0; t < kMT; ++t) {
      float x[8]; /* slot e: key 4 g + e, then 16 + 4 g + e - 4 */
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x[e] = s[t][e >> 2][e & 3] * a.scale_log2;
      }
      if (mask) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int key = b * kKeys + 16 * (e >> 2) + 4 * g + (e & 3);
          x[e] = key <= limit[t] ? x[e] : -INFINITY;
        }
      }
      float mx = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])),
                       fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
      mx = over_g_max(mx);
      /* The reference max moves only when a block's max passes it by more
       * than kSlack, and always from -inf. */
      const bool bump = mx > m_run[t] + kSlack;
      const float m_next = bump ? mx : m_run[t];
      const float m_use = m_next == -INFINITY ? 0.0f : m_next;
      float ps = 0.0f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float y = __builtin_fmaf(s[t][e >> 2][e & 3], a.scale_log2, -m_use);
        const float pe = __builtin_amdgcn_exp2f(y);
        x[e] = mask && x[e] == -INFINITY ? 0.0f : pe;
        ps += x[e];
      }
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        pt[t][w] = pack2(x[2 * w], x[2 * w + 1]);
      }
      const float alpha = bump ? __builtin_amdgcn_exp2f(m_run[t] - m_use) : 1.0f;
      l_run[t] = l_run[t] * alpha + ps;
      m_run[t] = m_next;
      if (__builtin_amdgcn_ballot_w64(bump) != 0) {
#pragma unroll
        for (int j = 0; j < kCols; ++j) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            o[t][j][r] *= alpha;
          }
        }
      }
    }
#pragma unroll
    for (int j = 0; j < kCols; ++j) {
      u32x4 vj;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        vj[d] = __builtin_amdgcn_perm(vf.f[2 * d + 1][j >> 1], vf.f[2 * d][j >> 1],
                                      j & 1 ? 0x07060302u : 0x05040100u);
      }
#pragma unroll
      for (int t = 0; t < kMT; ++t) {
        o[t][j] = mfma16<true>(vj, pt[t], o[t][j]);
      }
    }
    load_v(vf, b + 8);
  };

  Keys ka, kb;
  Values va, vb;
  load_k(ka, blk);
  load_v(va, blk);
  load_k(kb, blk + 4);
  load_v(vb, blk + 4);
  for (; blk < b1; blk += 8) {
    step(blk, ka, va);
    if (blk + 4 >= b1) {
      break;
    }
    step(blk + 4, kb, vb);
  }

  /* The four waves' results. o[t][j][r]: query 16 t + l16, d = kCols
   * (4 g + r) + j. */
  __shared__ float so[4][kRows][kPad];
  __shared__ float sm[4][kRows], sl[4][kRows];
#pragma unroll
  for (int t = 0; t < kMT; ++t) {
    const float l = over_g_sum(l_run[t]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
      for (int h = 0; h < kCols / 4; ++h) {
        *reinterpret_cast<f32x4 *>(&so[wave][16 * t + l16][kCols * (4 * g + r) + 4 * h]) =
            f32x4{o[t][4 * h][r], o[t][4 * h + 1][r], o[t][4 * h + 2][r], o[t][4 * h + 3][r]};
      }
    }
    if (g == 0) {
      sm[wave][16 * t + l16] = m_run[t];
      sl[wave][16 * t + l16] = l;
    }
  }
  __syncthreads();
  /* Thread: four columns of a row, kPer rows apart by kStep. */
  constexpr int kQuads = kD / 4;
  constexpr int kStep = kThreads / kQuads;
  constexpr int kPer = kRows / kStep;
  const int c4 = threadIdx.x % kQuads * 4;
  const int first = threadIdx.x / kQuads;
  f32x4 acc[kPer];
  float m[kPer], l[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int r = first + i * kStep;
    m[i] = fmaxf(fmaxf(sm[0][r], sm[1][r]), fmaxf(sm[2][r], sm[3][r]));
    const float m_use = m[i] == -INFINITY ? 0.0f : m[i];
    acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    l[i] = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = __builtin_amdgcn_exp2f(sm[w][r] - m_use); /* 0 where it saw none */
      l[i] += sl[w][r] * f;
      const f32x4 v = *reinterpret_cast<const f32x4 *>(&so[w][r][c4]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc[i][e] += v[e] * f;
      }
    }
  }
  if (p.splits > 1) {
    /* per split: [kRows][kD] outputs, then [kRows][2] max and sum */
    constexpr int kPart = kRows * (kD + 2) * 4;
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(p.ws + rows::kTicketBytes + (int64_t)item * p.splits * kPart), (short)0,
        p.splits * kPart, 0x00020000);
    __shared__ int last;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int r = first + i * kStep;
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[i]), wr,
                                             split * kPart + (r * kD + c4) * 4, 0, 16 /* sc1 */);
      if (c4 == 0) {
        __builtin_amdgcn_raw_buffer_store_b64(
            u32x2{__float_as_uint(m[i]), __float_as_uint(l[i])}, wr,
            split * kPart + (kRows * kD + 2 * r) * 4, 0, 16 /* sc1 */);
      }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    int *ticket = reinterpret_cast<int *>(p.ws) + item;
    if (threadIdx.x == 0) {
      const int n = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = n == p.splits - 1;
      if (n == p.splits - 1) { /* for the next launch */
        __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __syncthreads();
    if (!last) {
      return;
    }
    constexpr int kBatch = 4; /* splits' loads in flight, of every row */
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      m[i] = -INFINITY;
      l[i] = 0.0f;
      acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    for (int s0 = 0; s0 < p.splits; s0 += kBatch) {
      f32x4 v[kPer][kBatch];
      u32x2 ml[kPer][kBatch];
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int r = first + i * kStep;
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          const int at = (s0 + u) * kPart; /* zeros past the last split */
          v[i][u] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                  wr, at + (r * kD + c4) * 4, 0, 16 /* sc1 */));
          ml[i][u] = __builtin_bit_cast(
              u32x2, __builtin_amdgcn_raw_buffer_load_b64(wr, at + (kRows * kD + 2 * r) * 4, 0,
                                                          16 /* sc1 */));
        }
      }
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        float ms[kBatch], mx = m[i];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          ms[u] = s0 + u < p.splits ? __uint_as_float(ml[i][u][0]) : -INFINITY;
          mx = fmaxf(mx, ms[u]);
        }
        const float m_use = mx == -INFINITY ? 0.0f : mx;
        const float back = __builtin_amdgcn_exp2f(m[i] - m_use);
        l[i] *= back;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc[i][e] *= back;
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          const float f = __builtin_amdgcn_exp2f(ms[u] - m_use);
          l[i] += __uint_as_float(ml[i][u][1]) * f;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            acc[i][e] += v[i][u][e] * f;
          }
        }
        m[i] = mx;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int r = row0 + first + i * kStep;
    if (r >= a.rows) {
      continue;
    }
    const bool seen = l[i] > 0.0f;
    const float inv = seen ? 1.0f / l[i] : 0.0f;
    const int64_t at = kv * a.rows + r;
    *reinterpret_cast<u32x2 *>(a.o + at * kD + c4) =
        u32x2{pack2(acc[i][0] * inv, acc[i][1] * inv), pack2(acc[i][2] * inv, acc[i][3] * inv)};
    if (a.lse && c4 == 0) {
      a.lse[at] = seen ? (m[i] + log2f(l[i])) * 0.69314718055994531f : -INFINITY;
    }
  }
}

template <int kD, int kMT> void launch(const KernelArgs &p, hipStream_t stream) {
  hipLaunchKernelGGL((flash_rows<kD, kMT>),
                     dim3((unsigned)(p.a.kv_total * p.tiles * p.splits)), dim3(kThreads), 0,
                     stream, p);
}

template <int kD> void launch_mt(const KernelArgs &p, int mt, hipStream_t stream) {
  if (mt == 1) {
    launch<kD, 1>(p, stream);
  } else {
    launch<kD, 2>(p, stream);
  }
}

} // namespace

void flash_rows_launch(const rows::Args &a, const rows::Plan &plan, int head_dim, char *ws,
                       hipStream_t stream) {
  const KernelArgs p{a, plan.tiles, plan.splits, ws};
  if (head_dim == 128) {
    launch_mt<128>(p, plan.mt, stream);
  } else {
    launch_mt<64>(p, plan.mt, stream);
  }
}

} // namespace vxk
