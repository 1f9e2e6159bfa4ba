/*
 * gemm_ring.hip -- 16-bit GEMMs on 128x128 or 256x128 tiles, for grids that
 * leave many CUs without one of gemm.hip's 256x256 tiles.
 *
 * Waves of 64x64 on v_mfma_f32_16x16x32: four, two workgroups to a CU, or
 * eight, one to a CU (ring::tall). K in stages of 32 through an LDS ring (five
 * slots, or six) of buffer-to-LDS loads in the
 * layouts of the ping-pong kernel; a wave reads the next stage's operands
 * while it multiplies this one's, one barrier a stage. With `splits` > 1
 * several workgroups divide a tile's K: each leaves its sums in a workspace
 * past the caches that other XCDs do not see and takes a ticket; the one with
 * the last ticket adds them all in order and stores C.
 *
 * A stage takes 0.34 us where a CU has one workgroup and 0.53 where it has
 * two (690 TFLOP/s at 1024 x 4096 x 4096); what bounds it is getting 16 KiB a
 * stage and workgroup through L1 from L2 (the TCP waits on L2 60% of its
 * cycles, the matrix cores work 30% of a wave's time, no LDS read conflicts);
 * for 256x128, 24 KiB and 0.47 us, or 0.57 with B from HBM (TCP 38%, matrix
 * cores 44%). With four waves the larger tiles leave
 * the loads' latency open: 128x192 gave 67.5 us at 512 x 11008 x 4096 and 61 at
 * 1024 x 4096 x 4096 against 70.7 and 49, 256x128 78.8 and 70. Against the kernels
 * that took these shapes: 512 x 11008 x 4096 102 -> 76 us with
 * new inputs each pass (98 -> 66 on the same ones), 1024 x 4096 x 4096 66 -> 50, 2048^3 41 -> 28, 512 x 4096 x 11008 in 4 splits 77 -> 61 (in 1: 119).
 */
#include "../../../include/vx_hardware_runtime.h"
#include "../vx_hip_common.h"
#include "../vx_kernels.h"
#include "gemm_pp_layout.h"
#include "gemm_ring.h"
#include "vx_clock_stamp.hip.h"
#include "vx_lds_dma.hip.h"
#include "vx_mfma16.hip.h"

namespace vxk {
namespace {

typedef short i16x4 __attribute__((ext_vector_type(4)));

constexpr int kKs = 32; /* of k per stage */
constexpr int kBN = ring::kTile;
constexpr int kTM = 4, kTN = 4;  /* 16x16 blocks of a wave */
constexpr int kUB = kBN * 4;     /* 16-byte units per stage */
constexpr int kRowB = kBN / 8;   /* units per row of B */

template <int kOut> __device__ __forceinline__ void put4(void *c, int64_t at, f32x4 v, bool vec) {
  if constexpr (kOut == VX_DTYPE_F32) {
    float *p = static_cast<float *>(c) + at;
    if (vec) {
      *reinterpret_cast<f32x4 *>(p) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        p[e] = v[e];
      }
    }
  } else {
    uint32_t h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      h[e] = kOut == VX_DTYPE_BF16 ? f32_to_bf16(v[e]) : f32_to_f16(v[e]);
    }
    uint16_t *p = static_cast<uint16_t *>(c) + at;
    if (vec) {
      *reinterpret_cast<u32x2 *>(p) = u32x2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        p[e] = (uint16_t)h[e];
      }
    }
  }
}

template <bool kBf16, int kOut, int kBM, bool kStamp>
__global__ __launch_bounds__(2 * kBM, 2) void gemm_ring(
    const uint16_t *__restrict__ A, const uint16_t *__restrict__ B, void *__restrict__ C,
    int64_t M, int64_t N, int K, int64_t lda, int64_t ldb, int64_t ldc, int tiles_m,
    int tiles_n, int splits, char *__restrict__ ws, uint64_t *__restrict__ stamp) {
  const ClockStamp<kStamp> clocks(stamp);
  constexpr int kThreads = 2 * kBM;                         /* a wave per 64x64 */
  constexpr int kNS = kBM == 128 ? 5 : 6;                   /* slots: 80 KiB, or 144 */
  constexpr int kUA = kBM * 4;                              /* 16-byte units per stage */
  constexpr int kLA = kUA / kThreads, kLB = kUB / kThreads; /* loads per wave */
  constexpr int kPart = kBM * kBN * 4;                      /* bytes of a tile's sums */
  __shared__ u32x4 ring[kNS][kUA + kUB];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15;
  const int g = lane >> 4;
  const int wm = wave >> 1, wn = wave & 1;
  const int tiles = tiles_m * tiles_n;
  const int split = (int)blockIdx.x / tiles;
  const int id = (int)blockIdx.x - split * tiles;
  const pp::Tile tile = pp::tile_of(id, tiles, tiles_m, tiles_n);
  const int64_t m0 = (int64_t)tile.tm * kBM;
  const int64_t n0 = (int64_t)tile.tn * kBN;

  /* this workgroup's stages */
  const int all = K / kKs;
  const int first = (int)((int64_t)all * split / splits);
  const int stages = (int)((int64_t)all * (split + 1) / splits) - first;

  uint32_t a_off[kLA], b_off[kLB];
#pragma unroll
  for (int p = 0; p < kLA; ++p) {
    const int u = (wave * kLA + p) * 64 + lane;
    const int row = u >> 2;
    a_off[p] = (uint32_t)(row * lda * 2 + pp::dswz_a(row, u & 3) * 16);
  }
#pragma unroll
  for (int p = 0; p < kLB; ++p) {
    const int u = (wave * kLB + p) * 64 + lane;
    const int k = u / kRowB;
    b_off[p] = (uint32_t)(k * ldb * 2 + pp::pswz_b(k, u % kRowB) * 16);
  }
  /* Each stage's buffers end at the last element of their matrix: rows of A
   * past M and the tail of B's last row read zeros. Columns of B past N read
   * what follows, which only reaches columns of C that are not stored. */
  const int64_t a_end = ((M - 1) * lda + K) * 2, b_end = ((int64_t)(K - 1) * ldb + N) * 2;
  const uint32_t ring_base = (uint32_t)(uintptr_t)(VX_LDS void *)&ring[0][0];
  auto issue = [&](int st, int slot) {
    const int64_t a0 = (m0 * lda + (int64_t)(first + st) * kKs) * 2;
    const int64_t b0 = ((int64_t)(first + st) * kKs * ldb + n0) * 2;
    const int64_t a_full = (kBM - 1) * lda * 2 + kKs * 2, b_full = (kKs - 1) * ldb * 2 + kBN * 2;
    const i32x4 ra = buffer_rsrc((const char *)A + a0, (int)min(a_full, a_end - a0));
    const i32x4 rb = buffer_rsrc((const char *)B + b0, (int)min(b_full, b_end - b0));
    const uint32_t base = ring_base + (uint32_t)(slot * (kUA + kUB) * 16);
#pragma unroll
    for (int p = 0; p < kLA; ++p) {
      dma16(ra, a_off[p], base + (uint32_t)((wave * kLA + p) * 1024));
    }
#pragma unroll
    for (int p = 0; p < kLB; ++p) {
      dma16(rb, b_off[p], base + (uint32_t)(kUA * 16 + (wave * kLB + p) * 1024));
    }
  };

  struct Frags {
    u32x4 a[kTM], b[kTN];
  };
  auto read = [&](int slot, Frags &f) {
    const u32x4 *la = ring[slot];
    const VX_LDS char *lb = (const VX_LDS char *)&ring[slot][kUA];
#pragma unroll
    for (int j = 0; j < kTN; ++j) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int n = (wn * kTN + j) * 16 + 4 * (l16 & 3);
        const int k = 8 * g + 4 * h + (l16 >> 2);
        const int at = (k * kRowB + pp::pswz_b(k, n >> 3)) * 16 + (n & 7) * 2;
        const u32x2 w = __builtin_bit_cast(
            u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((VX_LDS i16x4 *)(lb + at)));
        f.b[j][2 * h] = w[0];
        f.b[j][2 * h + 1] = w[1];
      }
    }
#pragma unroll
    for (int i = 0; i < kTM; ++i) {
      const int row = (wm * kTM + i) * 16 + l16;
      f.a[i] = la[row * 4 + pp::dswz_a(row, g)];
    }
  };
  f32x4 acc[kTM][kTN];
#pragma unroll
  for (int i = 0; i < kTM; ++i) {
#pragma unroll
    for (int j = 0; j < kTN; ++j) {
      acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
  auto multiply = [&](const Frags &f) {
#pragma unroll
    for (int j = 0; j < kTN; ++j) {
#pragma unroll
      for (int i0 = 0; i0 < kTM; ++i0) {
        const int i = (j & 1) ? kTM - 1 - i0 : i0;
        acc[i][j] = mfma16<kBf16>(f.b[j], f.a[i], acc[i][j]);
      }
    }
  };

#pragma unroll
  for (int s = 0; s < kNS; ++s) {
    if (s < stages) {
      issue(s, s);
    }
  }
  wait_stages<kNS - 1, kLA + kLB>(min(stages, kNS) - 1);
  lds_barrier();
  Frags f0, f1;
  read(0, f0);
  /* Entering stage s: its operands are in `f`, and every wave's reads of them
   * end before the barrier, after which its slot takes stage s + kNS. The
   * next stage's reads run beside this one's MFMAs. */
  int slot = 0;
  auto stage = [&](int s, const Frags &f, Frags &next) {
    wait_stages<kNS - 2, kLA + kLB>(min(stages - 2 - s, kNS - 2));
    lds_barrier();
    if (s + kNS < stages) {
      issue(s + kNS, slot);
    }
    slot = slot == kNS - 1 ? 0 : slot + 1;
    read(slot, next);
    multiply(f);
  };
  int s = 0;
  for (; s + 2 < stages; s += 2) {
    stage(s, f0, f1);
    stage(s + 1, f1, f0);
  }
  if (s + 1 < stages) {
    stage(s, f0, f1);
    multiply(f1);
  } else {
    multiply(f0);
  }

  if (kBM == ring::kTile && splits > 1) {
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(ws + split::kTicketBytes + (int64_t)id * splits * kPart), (short)0,
        splits * kPart, 0x00020000);
    /* in the ring, whose reads are done after the barrier: with a word more
     * LDS than 80 KiB a CU has room for one workgroup only */
    int &last = *reinterpret_cast<int *>(&ring[0][0]);
    const int at = (int)threadIdx.x * 16;
#pragma unroll
    for (int i = 0; i < kTM; ++i) {
#pragma unroll
      for (int j = 0; j < kTN; ++j) {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[i][j]), wr,
                                               at + (i * kTN + j) * kThreads * 16,
                                               split * kPart, 16 /* sc1 */);
      }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    int *ticket = reinterpret_cast<int *>(ws) + id;
    if (threadIdx.x == 0) {
      const int n = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = n == splits - 1;
      if (n == splits - 1) { /* for the next launch */
        __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __syncthreads();
    if (!last) {
      clocks.end();
      return;
    }
    for (int s2 = 0; s2 < splits; ++s2) {
      f32x4 v[kTM][kTN];
#pragma unroll
      for (int i = 0; i < kTM; ++i) {
#pragma unroll
        for (int j = 0; j < kTN; ++j) {
          v[i][j] = __builtin_bit_cast(
              f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                         wr, at + (i * kTN + j) * kThreads * 16, s2 * kPart, 16 /* sc1 */));
        }
      }
#pragma unroll
      for (int i = 0; i < kTM; ++i) {
#pragma unroll
        for (int j = 0; j < kTN; ++j) {
          acc[i][j] = s2 == 0 ? v[i][j] : acc[i][j] + v[i][j];
        }
      }
    }
  }

  const bool vec = (ldc & 3) == 0 && ((uintptr_t)C & (kOut == VX_DTYPE_F32 ? 15 : 7)) == 0;
#pragma unroll
  for (int i = 0; i < kTM; ++i) {
#pragma unroll
    for (int j = 0; j < kTN; ++j) {
      const int64_t row = m0 + (wm * kTM + i) * 16 + l16;
      const int64_t col = n0 + (wn * kTN + j) * 16 + 4 * g;
      if (row < M && col < N) {
        put4<kOut>(C, row * ldc + col, acc[i][j], vec);
      }
    }
  }
  clocks.end();
}

template <bool kBf16, int kOut, int kBM>
void launch_rows(const GemmArgs &g, int splits, char *ws, hipStream_t s) {
  const int tiles_m = (int)((g.m + kBM - 1) / kBM), tiles_n = (int)((g.n + kBN - 1) / kBN);
  const auto kernel = g.stamp ? gemm_ring<kBf16, kOut, kBM, true> : gemm_ring<kBf16, kOut, kBM, false>;
  hipLaunchKernelGGL(kernel, dim3(tiles_m * tiles_n * splits), dim3(2 * kBM), 0, s,
                     static_cast<const uint16_t *>(g.a), static_cast<const uint16_t *>(g.b),
                     g.c, g.m, g.n, (int)g.k, g.lda, g.ldb, g.ldc, tiles_m, tiles_n, splits, ws,
                     g.stamp);
}

template <bool kBf16, int kOut>
void launch(const GemmArgs &g, int splits, char *ws, hipStream_t s) {
  if (splits == 1 && ring::tall(g.m, g.n, g.k, device_cu_count())) {
    launch_rows<kBf16, kOut, 2 * ring::kTile>(g, 1, nullptr, s);
  } else {
    launch_rows<kBf16, kOut, ring::kTile>(g, splits, ws, s);
  }
}

} // namespace

void gemm_ring_launch(const GemmArgs &g, int splits, char *ws, hipStream_t s) {
  const bool bf = g.in_dtype == VX_DTYPE_BF16;
  if (g.out_dtype == VX_DTYPE_F32) {
    bf ? launch<true, VX_DTYPE_F32>(g, splits, ws, s) : launch<false, VX_DTYPE_F32>(g, splits, ws, s);
  } else if (bf) {
    launch<true, VX_DTYPE_BF16>(g, splits, ws, s);
  } else {
    launch<false, VX_DTYPE_F16>(g, splits, ws, s);
  }
}

} // namespace vxk
