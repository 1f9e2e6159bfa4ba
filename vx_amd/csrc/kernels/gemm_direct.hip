/*
 * gemm_direct.hip -- 16-bit GEMMs whose operands go straight from memory
 * into MFMA registers: few rows, shapes and row strides off the 16-byte grid,
 * and grids too small for the 256x256 tiles of gemm.hip.
 *
 * A wave owns 16 kMT rows x 128 columns of C. For each 32 of k a lane loads
 * eight 16-byte pieces of B, rows k = 8 g .. 8 g + 7 (g = lane / 16) of its
 * own eight columns, and turns that 8 x 8 block in registers (32 v_perm)
 * into the operands of eight MFMAs, one per column of the eight; A's operand
 * is 16 bytes of a row as they lie. So nothing passes through LDS, a load
 * covers 256 contiguous bytes of B, and no address has to be aligned beyond
 * the element. The lane ends up with eight consecutive columns of a row of C.
 * What bounds it is the load path into the registers (12 KiB a wave for 64 x
 * 128 x 32 multiply-adds), and for few rows reading B.
 *
 * bf16 -> f32, against the kernels that took these shapes before (scalar
 * exact-order, or 256x256 tiles): 8 x 4096 x 4096 178 -> 8.0 us (4.2 TB/s of
 * B), f16 1000 x 777 x 1111 117 -> 12.9, 512 x 4096 x 4096 88 -> 33, 1024^3
 * 29 -> 8.4, 4000 x 4001 x 3999 (odd rows) 328 us, 390 TFLOP/s.
 *
 * kAlongK: the four waves of a workgroup take the same tile and a quarter of
 * k each, and add up in LDS; with `splits` > 1 so do several workgroups, in
 * a workspace: each leaves its sums and takes a ticket, and the one with the
 * last ticket adds all of them in order, so the result does not depend on
 * who is last and nobody waits. Otherwise the four waves stand below each
 * other, sharing B through L1, each over all of k.
 */
#include "../../../include/vx_hardware_runtime.h"
#include "../vx_hip_common.h"
#include "../vx_kernels.h"
#include "gemm_direct.h"
#include "vx_clock_stamp.hip.h"
#include "vx_mfma16.hip.h"

#include <algorithm>

namespace vxk {
namespace {

constexpr int kThreads = 256;
constexpr int kCols = 128; /* of C per wave */

/* 16 bytes from any 2-byte boundary. */
struct __attribute__((packed, aligned(2))) Any16 {
  u32x4 v;
};
__device__ __forceinline__ u32x4 load16(const char *p) {
  return reinterpret_cast<const Any16 *>(p)->v;
}

struct DirectArgs {
  const char *a, *b;
  char *c;
  int64_t lda, ldb, ldc;
  int64_t m, n;
  int k;
  int tiles_m, tiles_n;
  int splits;
  char *ws;
  uint64_t *stamp;
};

/* Eight consecutive columns of a row of C. */
template <int kOut> __device__ __forceinline__ void put8(char *c, int64_t at, const float (&v)[8]) {
  if constexpr (kOut == VX_DTYPE_F32) {
    char *p = c + at * 4;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      reinterpret_cast<Any16 *>(p)[h].v = __builtin_bit_cast(
          u32x4, f32x4{v[4 * h], v[4 * h + 1], v[4 * h + 2], v[4 * h + 3]});
    }
  } else {
    u32x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t lo = kOut == VX_DTYPE_BF16 ? f32_to_bf16(v[2 * e]) : f32_to_f16(v[2 * e]);
      const uint32_t hi =
          kOut == VX_DTYPE_BF16 ? f32_to_bf16(v[2 * e + 1]) : f32_to_f16(v[2 * e + 1]);
      w[e] = lo | (hi << 16);
    }
    reinterpret_cast<Any16 *>(c + at * 2)->v = w;
  }
}

template <bool kBf16, int kOut, int kMT, int kBuf, bool kAlongK, bool kOddA, bool kStamp>
__global__ __launch_bounds__(kThreads, kMT <= 2 ? 2 : 1) void gemm_direct(DirectArgs p) {
  const ClockStamp<kStamp> clocks(p.stamp);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15;
  const int g = lane >> 4;

  /* Workgroup -> (split, tile). Consecutive ids lie on different XCDs: give
   * each XCD a run of tiles, the rows of a column of tiles first, whose B
   * its L2 then holds. */
  int id = blockIdx.x;
  if ((gridDim.x & 7) == 0) {
    id = (id & 7) * (int)(gridDim.x >> 3) + (id >> 3);
  }
  const int tiles = p.tiles_m * p.tiles_n;
  const int split = kAlongK ? id % p.splits : 0;
  const int tile = kAlongK ? id / p.splits : id;
  const int64_t m0 = (int64_t)(tile % p.tiles_m) * (16 * kMT * (kAlongK ? 1 : 4)) +
                     (kAlongK ? 0 : wave * 16 * kMT);
  const int64_t n0 = (int64_t)(tile / p.tiles_m) * kCols;
  if (!kAlongK && m0 >= p.m) {
    return;
  }

  /* This wave's blocks of 32 k. */
  const int nb = (p.k + 31) / 32, whole = p.k / 32;
  const int parts = kAlongK ? 4 * p.splits : 1;
  const int part = kAlongK ? 4 * split + wave : 0;
  const int b0 = (int)((int64_t)nb * part / parts);
  const int b1 = (int)((int64_t)nb * (part + 1) / parts);
  const int fb = min(b1, whole);

  /* The lane's eight columns start at n0 + 8 l16, moved back where they would
   * run past the last (a column that two lanes then hold gets the same value
   * from both). Rows past the last read the last. */
  const int64_t col = min(n0 + 8 * l16, p.n - 8);
  uint32_t boff[8], aoff[kMT];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    boff[i] = (uint32_t)(((8 * g + i) * p.ldb + (col - min(n0, p.n - 8))) * 2);
  }
  const char *bb = p.b + min(n0, p.n - 8) * 2;
  const char *ab = p.a + m0 * p.lda * 2;
  /* kOddA: a row of A may start on any element. A 16-byte load off the
   * 4-byte grid takes several times as long, so each lane loads the words
   * that hold its piece, the fifth of them only where the piece starts inside
   * the first, and shifts. Each word holds an element of the row. */
  const uint32_t odd = kOddA ? (uint32_t)(uintptr_t)ab & 2 : 0;
  ab -= odd;
  uint32_t ashift[kMT];
#pragma unroll
  for (int t = 0; t < kMT; ++t) {
    aoff[t] = (uint32_t)((min(m0 + 16 * t + l16, p.m - 1) - m0) * p.lda * 2 + 16 * g) + odd;
    ashift[t] = kOddA ? 8 * (aoff[t] & 2) : 0;
  }

  struct Block {
    u32x4 b[8], a[kMT];
    uint32_t a4[kOddA ? kMT : 1];
  };
  f32x4 acc[kMT][8];
#pragma unroll
  for (int t = 0; t < kMT; ++t) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      acc[t][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
  auto load = [&](Block &f, int blk) {
    const char *bp = bb + (int64_t)blk * 32 * p.ldb * 2;
    const char *ap = ab + (int64_t)blk * 64;
#pragma unroll
    for (int t = 0; t < kMT; ++t) {
      if constexpr (kOddA) {
        const char *words = ap + (aoff[t] & ~3u);
        f.a[t] = load16(words);
        f.a4[t] = *reinterpret_cast<const uint32_t *>(words + 12 + ashift[t] / 4);
      } else {
        f.a[t] = load16(ap + aoff[t]);
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      f.b[i] = load16(bp + boff[i]);
    }
  };
  auto multiply = [&](const u32x4 (&b)[8], const u32x4 (&a)[kMT]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      u32x4 bj;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        bj[d] = __builtin_amdgcn_perm(b[2 * d + 1][j >> 1], b[2 * d][j >> 1],
                                      j & 1 ? 0x07060302u : 0x05040100u);
      }
#pragma unroll
      for (int t = 0; t < kMT; ++t) {
        acc[t][j] = mfma16<kBf16>(bj, a[t], acc[t][j]);
      }
    }
  };
  auto compute = [&](const Block &f) {
    if constexpr (kOddA) {
      u32x4 a[kMT];
#pragma unroll
      for (int t = 0; t < kMT; ++t) {
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          a[t][d] = __builtin_amdgcn_alignbit(d < 3 ? f.a[t][d + 1] : f.a4[t], f.a[t][d],
                                              ashift[t]);
        }
      }
      multiply(f.b, a);
    } else {
      multiply(f.b, f.a);
    }
  };

  Block f[kBuf];
  int blk = b0;
  if (fb - b0 >= kBuf) {
#pragma unroll
    for (int s = 0; s < kBuf; ++s) {
      load(f[s], blk + s);
    }
    for (; blk + 2 * kBuf <= fb; blk += kBuf) {
#pragma unroll
      for (int s = 0; s < kBuf; ++s) {
        compute(f[s]);
        load(f[s], blk + kBuf + s);
      }
    }
#pragma unroll
    for (int s = 0; s < kBuf; ++s) {
      compute(f[s]);
    }
    blk += kBuf;
  }
  /* fewer than kBuf blocks are left */
#pragma unroll
  for (int s = 0; s < kBuf - 1; ++s) {
    if (blk + s < fb) {
      load(f[s], blk + s);
    }
  }
#pragma unroll
  for (int s = 0; s < kBuf - 1; ++s) {
    if (blk + s < fb) {
      compute(f[s]);
    }
  }
  if (b1 > whole) {
    /* the last k, fewer than 32: zeros past them on both sides */
    Block &t = f[0];
    const char *bp = bb + (int64_t)whole * 32 * p.ldb * 2;
    const char *ap = ab + (int64_t)whole * 64;
    const int left = p.k - 32 * whole;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      t.b[i] = u32x4{0, 0, 0, 0};
      if (8 * g + i < left) {
        t.b[i] = load16(bp + boff[i]);
      }
    }
#pragma unroll
    for (int r = 0; r < kMT; ++r) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t w = 0;
        if (8 * g + 2 * e < left) {
          w = reinterpret_cast<const uint16_t *>(ap + aoff[r])[2 * e];
        }
        if (8 * g + 2 * e + 1 < left) {
          w |= (uint32_t)reinterpret_cast<const uint16_t *>(ap + aoff[r])[2 * e + 1] << 16;
        }
        t.a[r][e] = w;
      }
    }
    multiply(t.b, t.a);
  }

  /* acc[t][j][r]: row 16 t + l16, the j-th of the eight columns of group
   * 4 g + r (the columns that lane 4 g + r of 16 loaded). */
  auto store = [&](int t, int r, const float (&v)[8]) {
    const int64_t row = m0 + 16 * t + l16;
    const int64_t c0 = n0 + 8 * (4 * g + r);
    if (row < p.m && c0 < p.n) {
      put8<kOut>(p.c, row * p.ldc + min(c0, p.n - 8), v);
    }
  };
  if constexpr (!kAlongK) {
#pragma unroll
    for (int t = 0; t < kMT; ++t) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          v[j] = acc[t][j][r];
        }
        store(t, r, v);
      }
    }
    clocks.end();
    return;
  }

  /* Piece q = 2 (4 t + r) + h: columns 4 h .. 4 h + 3 of the eight. Wave w
   * adds the pieces of 4 t + r = w kMT .. w kMT + kMT - 1. */
  __shared__ f32x4 red[4][8 * kMT][64];
#pragma unroll
  for (int t = 0; t < kMT; ++t) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        red[wave][2 * (4 * t + r) + h][lane] =
            f32x4{acc[t][4 * h][r], acc[t][4 * h + 1][r], acc[t][4 * h + 2][r],
                  acc[t][4 * h + 3][r]};
      }
    }
  }
  __syncthreads();
  f32x4 own[2 * kMT];
#pragma unroll
  for (int q = 0; q < 2 * kMT; ++q) {
    const int at = wave * 2 * kMT + q;
    own[q] = (red[0][at][lane] + red[1][at][lane]) + (red[2][at][lane] + red[3][at][lane]);
  }
  if (p.splits > 1) {
    /* The partial sums and the ticket bypass the caches that other XCDs do
     * not see (sc1); each wave's stores are there before the barrier, and so
     * before the ticket. */
    constexpr int kPart = 8 * kMT * 64 * 16; /* bytes of one split's sums of a tile */
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(p.ws + split::kTicketBytes + (int64_t)tile * p.splits * kPart), (short)0,
        p.splits * kPart, 0x00020000);
    const int at = (wave * 2 * kMT * 64 + lane) * 16;
#pragma unroll
    for (int q = 0; q < 2 * kMT; ++q) {
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, own[q]), wr, at + q * 1024,
                                             split * kPart, 16 /* sc1 */);
    }
    __shared__ int last;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    int *ticket = reinterpret_cast<int *>(p.ws) + tile;
    if (threadIdx.x == 0) {
      const int n = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = n == p.splits - 1;
      if (n == p.splits - 1) { /* for the next launch */
        __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __syncthreads();
    if (!last) {
      clocks.end();
      return;
    }
    f32x4 sum[2 * kMT];
    for (int s = 0; s < p.splits; s += 4) {
      f32x4 v[4][2 * kMT];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
#pragma unroll
        for (int q = 0; q < 2 * kMT; ++q) { /* zeros past the last split */
          v[u][q] = __builtin_bit_cast(
              f32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, at + q * 1024 + (s + u) * kPart, 0,
                                                           16 /* sc1 */));
        }
      }
#pragma unroll
      for (int q = 0; q < 2 * kMT; ++q) {
        const f32x4 four = (v[0][q] + v[1][q]) + (v[2][q] + v[3][q]);
        sum[q] = s == 0 ? four : sum[q] + four;
      }
    }
#pragma unroll
    for (int q = 0; q < 2 * kMT; ++q) {
      own[q] = sum[q];
    }
  }
#pragma unroll
  for (int i = 0; i < kMT; ++i) {
    const int tr = wave * kMT + i;
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[j] = own[2 * i + (j >> 2)][j & 3];
    }
    store(tr >> 2, tr & 3, v);
  }
  clocks.end();
}

/* kBuf blocks of a wave's loads in flight, as its registers allow: kBufOdd for
 * an A off the 4-byte grid, which takes a word more a row. Two blocks at 32
 * rows, with two workgroups to a CU, against three and one: 256 x 4096 x 4096
 * 20.7 and 23.1 us. Eight waves a workgroup instead of four: no gain (64 x
 * 4096 x 4096 11.4 and 12.2, 1000 x 777 x 1111 13.1 and 12.9). */
template <bool kBf16, int kOut, int kMT, int kBuf, int kBufOdd, bool kAlongK>
void launch(const DirectArgs &p, hipStream_t s) {
  const bool odd = (p.lda & 1) || (reinterpret_cast<uintptr_t>(p.a) & 2);
  const auto kernel = odd ? p.stamp ? gemm_direct<kBf16, kOut, kMT, kBufOdd, kAlongK, true, true>
                                    : gemm_direct<kBf16, kOut, kMT, kBufOdd, kAlongK, true, false>
                      : p.stamp ? gemm_direct<kBf16, kOut, kMT, kBuf, kAlongK, false, true>
                                : gemm_direct<kBf16, kOut, kMT, kBuf, kAlongK, false, false>;
  hipLaunchKernelGGL(kernel, dim3(p.tiles_m * p.tiles_n * p.splits), dim3(kThreads), 0, s, p);
}

template <bool kBf16, int kOut>
void launch_plan(const DirectArgs &p, const direct::Plan &plan, hipStream_t s) {
  if (!plan.along_k) {
    launch<kBf16, kOut, 4, 2, 2, false>(p, s);
  } else if (plan.mt == 1) {
    launch<kBf16, kOut, 1, 4, 3, true>(p, s);
  } else if (plan.mt == 2) {
    launch<kBf16, kOut, 2, 2, 2, true>(p, s);
  } else {
    launch<kBf16, kOut, 4, 2, 2, true>(p, s);
  }
}

} // namespace

bool gemm_direct_takes(const GemmArgs &g) {
  const bool sixteen = g.in_dtype == VX_DTYPE_BF16 || g.in_dtype == VX_DTYPE_F16;
  const bool out_ok = g.out_dtype == VX_DTYPE_F32 || g.out_dtype == g.in_dtype;
  const uintptr_t low = reinterpret_cast<uintptr_t>(g.a) | reinterpret_cast<uintptr_t>(g.b);
  const uintptr_t c_low = reinterpret_cast<uintptr_t>(g.c);
  return sixteen && out_ok && (low & 1) == 0 && (c_low & (g.out_dtype == VX_DTYPE_F32 ? 3 : 1)) == 0 &&
         direct::shape_ok(g.m, g.n, g.k, g.lda, g.ldb, g.ldc);
}

void gemm_direct_launch(const GemmArgs &g, const direct::Plan &plan, char *ws, hipStream_t s) {
  DirectArgs p;
  p.a = static_cast<const char *>(g.a);
  p.b = static_cast<const char *>(g.b);
  p.c = static_cast<char *>(g.c);
  p.lda = g.lda, p.ldb = g.ldb, p.ldc = g.ldc;
  p.m = g.m, p.n = g.n, p.k = (int)g.k;
  p.tiles_m = plan.tiles_m, p.tiles_n = plan.tiles_n, p.splits = plan.splits;
  p.ws = ws;
  p.stamp = g.stamp;
  const bool bf = g.in_dtype == VX_DTYPE_BF16;
  if (g.out_dtype == VX_DTYPE_F32) {
    bf ? launch_plan<true, VX_DTYPE_F32>(p, plan, s) : launch_plan<false, VX_DTYPE_F32>(p, plan, s);
  } else if (bf) {
    launch_plan<true, VX_DTYPE_BF16>(p, plan, s);
  } else {
    launch_plan<false, VX_DTYPE_F16>(p, plan, s);
  }
}

} // namespace vxk
