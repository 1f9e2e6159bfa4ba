/*
 * gemm_f32.hip -- f32 GEMM for products large enough that the exact-order
 * kernel's rate matters, on bf16 MFMAs.
 *
 * An f32 value is the exact sum of three bf16 values, its 24 significant bits
 * 8 at a time, and the product of two such values is exact in f32. Of the nine
 * products of a pair the six of up to 2^-16 of the largest are added (the rest
 * are below 2^-24 of it, under the rounding of the f32 sums): the large ones
 * in one accumulator, the other five in a second, added at the end. Six
 * v_mfma_f32_16x16x32_bf16 do 32 of k in 96 cycles; f32 MFMAs take 256.
 * Infinities, and rows of A or columns of B without a value of 2^-100 or
 * more, whose last bits bf16 cannot hold, are left to f32 MFMAs: a tile that
 * met one is computed again that way. (A NaN passes through the planes.)
 *
 * 128 x 128 tiles, eight waves of 64 x 32, K in stages of 32 through two LDS
 * slots. A thread loads 8 k of one row of A and of one column of B, splits
 * them between the MFMAs of the stage before, and writes each plane's 16
 * bytes as the MFMA operands want them: [row][chunk of 8 k], chunks XORed so
 * that 16 rows at one chunk lie in distinct banks, for the reads and both
 * writes; three stages' loads are in flight (with two: 1999 x 2001 x 2003 107
 * us against 98, 300 x 4000 x 4096 163 against 150). What bounds it: at 2048^3
 * the matrix cores work 45% of the cycles, at 2.1 GHz under their load; a
 * stage's operand reads (144 KiB) and its MFMAs follow one another between
 * barriers (taking a SIMD's two waves in turns, one reading while the other
 * multiplies, costs a barrier more and gave the same: 108 us).
 *
 * Against f32 MFMAs in the same tile: 2048^3 248 -> 92 us with new inputs each
 * pass (188 TFLOP/s), 258 -> 104 with the same ones; error against 64 bits
 * 8.1e-7 -> 2.5e-7 at 2048^3, 1.1e-6 -> 3.8e-7 at K = 4096. Grids of fewer
 * tiles than CUs divide K over workgroups: 1024^3 125 -> 27 us (undivided 45),
 * 128 x 4096 x 4096 454 -> 38 (142).
 */
#include "../vx_hip_common.h"
#include "../vx_kernels.h"
#include "gemm_f32.h"
#include "gemm_pp_layout.h"
#include "vx_lds_dma.hip.h"
#include "vx_mfma16.hip.h"

namespace vxk {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kThreads = 512;
constexpr int kTile = f32::kTile;
constexpr int kKs = 32;               /* of k per stage */
constexpr int kPlane = kTile * 4;     /* 16-byte units */
constexpr float kLeast = 7.888609052210118e-31f; /* 2^-100 */

struct __attribute__((packed, aligned(4))) Four {
  f32x4 v;
};

struct Regs {
  float a[8], b[8];
};

__device__ __forceinline__ int unit(int row, int c) { return row * 4 + (c ^ ((row >> 1) & 3)); }

/* Eight values as the three planes' 16 bytes. */
__device__ __forceinline__ void split8(const float (&x)[8], u32x4 (&p)[3]) {
  uint32_t u[8], r[8], s[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    u[e] = __float_as_uint(x[e]);
    const float d = x[e] - __uint_as_float(u[e] & 0xffff0000u);
    r[e] = __float_as_uint(d);
    s[e] = __float_as_uint(d - __uint_as_float(r[e] & 0xffff0000u));
  }
#pragma unroll
  for (int w = 0; w < 4; ++w) { /* upper halves */
    p[0][w] = __builtin_amdgcn_perm(u[2 * w + 1], u[2 * w], 0x07060302u);
    p[1][w] = __builtin_amdgcn_perm(r[2 * w + 1], r[2 * w], 0x07060302u);
    p[2][w] = __builtin_amdgcn_perm(s[2 * w + 1], s[2 * w], 0x07060302u);
  }
}

__global__ __launch_bounds__(kThreads, 2) void gemm_f32_mfma(
    const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ C, int64_t M,
    int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int tiles_m, int tiles_n,
    int splits, char *__restrict__ ws) {
  __shared__ u32x4 lds[2][2][3][kPlane]; /* [slot][A, B][plane] */
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int l16 = lane & 15;
  const int g = lane >> 4;
  const int wm = wave >> 2, wn = wave & 3;
  const int tiles = tiles_m * tiles_n;
  const int split = (int)blockIdx.x / tiles;
  const int id = (int)blockIdx.x - split * tiles;
  const pp::Tile tile = pp::tile_of(id, tiles, tiles_m, tiles_n);
  const int64_t m0 = (int64_t)tile.tm * kTile;
  const int64_t n0 = (int64_t)tile.tn * kTile;

  /* Thread: row t / 4 of A at chunk t % 4; column t % 128 of B at chunk
   * t / 128. Rows and columns past the last read the last. */
  const int a_row = t >> 2, a_chunk = t & 3;
  const int b_col = t & 127;
  const int b_chunk = wave >> 1;
  /* this workgroup's stages */
  const int64_t all = (K + kKs - 1) / kKs;
  const int64_t first = all * split / splits;
  const int64_t stages = all * (split + 1) / splits - first;
  const int64_t whole = min(first + stages, K / kKs) - first;
  const int64_t left = K - first * kKs; /* k from its first on */
  const float *pa = A + min(m0 + a_row, M - 1) * lda + first * kKs + 8 * a_chunk;
  const int b_off = (int)(min(n0 + b_col, N - 1) - n0);
  const float *pb = B + (first * kKs + 8 * b_chunk) * ldb + n0;

  auto load = [&](Regs &r, int64_t st) {
    const float *a = pa + st * kKs;
    const float *b = pb + st * kKs * ldb;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4 v = reinterpret_cast<const Four *>(a)[h].v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        r.a[4 * h + e] = v[e];
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      r.b[e] = (b + e * ldb)[b_off];
    }
  };
  auto load_last = [&](Regs &r, int64_t st) { /* zeros past K */
    const float *a = pa + st * kKs;
    const float *b = pb + st * kKs * ldb;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      r.a[e] = st * kKs + 8 * a_chunk + e < left ? a[e] : 0.0f;
      r.b[e] = st * kKs + 8 * b_chunk + e < left ? (b + e * ldb)[b_off] : 0.0f;
    }
  };
  float a_max = 0.0f, b_max = 0.0f; /* of the row's and column's magnitudes */
  auto stash = [&](const Regs &r, int slot) {
    u32x4 p[3];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      a_max = fmaxf(a_max, __builtin_fabsf(r.a[e]));
      b_max = fmaxf(b_max, __builtin_fabsf(r.b[e]));
    }
    split8(r.a, p);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      lds[slot][0][i][unit(a_row, a_chunk)] = p[i];
    }
    split8(r.b, p);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      lds[slot][1][i][unit(b_col, b_chunk)] = p[i];
    }
  };

  /* hi, lo[i][j]: rows 64 wm + 16 i + l16, columns 32 wn + 16 j + 4 g .. + 3 */
  f32x4 hi[4][2], lo[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      hi[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      lo[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
  u32x4 af[3][4], bf[3][2];
  auto fragments = [&](int slot) {
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        bf[p][j] = lds[slot][1][p][unit(32 * wn + 16 * j + l16, g)];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        af[p][i] = lds[slot][0][p][unit(64 * wm + 16 * i + l16, g)];
      }
    }
  };
  auto multiply = [&]() {
    auto add = [&](int pa_, int pb_, f32x4 (&c)[4][2]) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          c[i][j] = mfma16<true>(bf[pb_][j], af[pa_][i], c[i][j]);
        }
      }
    };
    add(0, 0, hi);
    add(0, 1, lo);
    add(1, 0, lo);
    add(1, 1, lo);
    add(0, 2, lo);
    add(2, 0, lo);
  };

  auto load_any = [&](Regs &r, int64_t st) {
    if (st < whole) {
      load(r, st);
    } else {
      load_last(r, st);
    }
  };
  /* Entering stage s: it is in slot s % 2, the next in r[(s + 1) % 3], the one
   * after in r[(s + 2) % 3]. */
  Regs r[3];
  load_any(r[0], 0);
  if (stages > 1) {
    load_any(r[1], 1);
  }
  if (stages > 2) {
    load_any(r[2], 2);
  }
  stash(r[0], 0);
  lds_barrier();
  int64_t st = 0;
  auto stage = [&](int64_t s, int slot, const Regs &next, Regs &after) {
    load(after, s + 3);
    fragments(slot);
    multiply();
    stash(next, slot ^ 1);
#pragma unroll
    for (int i = 0; i < 48; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); /* MFMA */
      __builtin_amdgcn_sched_group_barrier(0x002, 3, 0); /* VALU */
    }
    lds_barrier();
  };
  for (; st + 8 < whole; st += 6) {
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      stage(st + i, i & 1, r[(i + 1) % 3], r[i % 3]);
    }
  }
  for (; st < stages; ++st) {
    const int slot = (int)(st & 1);
    fragments(slot);
    if (st + 1 < stages) {
      stash(r[1], slot ^ 1);
    }
    r[1] = r[2];
    if (st + 3 < stages) {
      load_any(r[2], st + 3);
    }
    multiply();
    lds_barrier();
  }

  /* The row's other three threads are its lane's neighbours, the column's
   * other three in other waves. */
  auto odd = [&](float v) { return !(v < INFINITY) || (v > 0.0f && v < kLeast); };
#pragma unroll
  for (int o = 1; o < 4; o *= 2) {
    a_max = fmaxf(a_max, __shfl_xor(a_max, o));
  }
  float *cols = reinterpret_cast<float *>(&lds[0][0][0][0]); /* [4][128] */
  cols[b_chunk * kTile + b_col] = b_max;
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    b_max = fmaxf(b_max, cols[c * kTile + b_col]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        hi[i][j][e] = hi[i][j][e] + lo[i][j][e];
      }
    }
  }
  if (splits > 1) {
    /* The sums, then the magnitudes, go past the caches that other XCDs do not
     * see; the workgroup with the last ticket adds all of them up in order. */
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(ws + f32::kTicketBytes + (int64_t)id * splits * f32::kPart), (short)0,
        splits * f32::kPart, 0x00020000);
    constexpr int kMax = kTile * kTile * 4; /* [128] of the rows, [128] of the columns */
    const int at = t * 16;
    __shared__ int last;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, hi[i][j]), wr,
                                               at + (2 * i + j) * kThreads * 16,
                                               split * f32::kPart, 16 /* sc1 */);
      }
    }
    if (a_chunk == 0) {
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(a_max), wr, kMax + a_row * 4,
                                            split * f32::kPart, 16 /* sc1 */);
    }
    if (b_chunk == 0) {
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(b_max), wr,
                                            kMax + (kTile + b_col) * 4, split * f32::kPart,
                                            16 /* sc1 */);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    int *ticket = reinterpret_cast<int *>(ws) + id;
    if (t == 0) {
      const int n = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = n == splits - 1;
      if (n == splits - 1) { /* for the next launch */
        __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __syncthreads();
    if (!last) {
      return;
    }
    a_max = b_max = 0.0f;
    for (int s = 0; s < splits; ++s) {
      f32x4 v[4][2];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          v[i][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                  wr, at + (2 * i + j) * kThreads * 16,
                                                  s * f32::kPart, 16 /* sc1 */));
        }
      }
      a_max = fmaxf(a_max, __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                               wr, kMax + a_row * 4, s * f32::kPart, 16 /* sc1 */)));
      b_max = fmaxf(b_max, __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                               wr, kMax + (kTile + b_col) * 4, s * f32::kPart, 16 /* sc1 */)));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          hi[i][j] = s == 0 ? v[i][j] : hi[i][j] + v[i][j];
        }
      }
    }
  }
  if (!__syncthreads_or(odd(a_max) || odd(b_max))) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int64_t row = m0 + 64 * wm + 16 * i + l16;
        const int64_t col = n0 + 32 * wn + 16 * j + 4 * g;
        if (row < M && col < N) {
          float *c = C + row * ldc + col;
          if (col + 3 < N) {
            reinterpret_cast<Four *>(c)->v = hi[i][j];
          } else {
#pragma unroll
            for (int e = 0; e < 3; ++e) {
              if (col + e < N) {
                c[e] = hi[i][j][e];
              }
            }
          }
        }
      }
    }
    return;
  }

  /* The tile again on v_mfma_f32_32x32x2_f32: stages of 16 of k through one
   * LDS slot, operands as [k][m] and [k][n] with 32 floats between the two
   * half-waves' rows. */
  constexpr int kFs = 16, kPad = kTile + 32;
  float(*as)[kPad] = reinterpret_cast<float(*)[kPad]>(&lds[0][0][0][0]);
  float(*bs)[kPad] = as + kFs;
  f32x16 acc[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc[i][r] = 0.0f;
    }
  }
  const int64_t am = min(m0 + (t >> 2), M - 1), bn0 = n0 + 4 * (t & 31);
  const int ak = 4 * (t & 3), bk = t >> 5;
  for (int64_t k0 = 0; k0 < K; k0 += kFs) {
    float ra[4], rb[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      ra[e] = k0 + ak + e < K ? A[am * lda + k0 + ak + e] : 0.0f;
      rb[e] = k0 + bk < K ? B[(k0 + bk) * ldb + min(bn0 + e, N - 1)] : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      as[ak + e][t >> 2] = ra[e];
      bs[bk][4 * (t & 31) + e] = rb[e];
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < kFs; kk += 2) {
      const float b = bs[kk + (lane >> 5)][32 * wn + (lane & 31)];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float a = as[kk + (lane >> 5)][64 * wm + 32 * i + (lane & 31)];
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[i], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int64_t col = n0 + 32 * wn + (lane & 31);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int64_t row = m0 + 64 * wm + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
      if (row < M && col < N) {
        C[row * ldc + col] = acc[i][r];
      }
    }
  }
}

} // namespace

void gemm_f32_launch(const GemmArgs &g, int splits, char *ws, hipStream_t s) {
  const int tiles_m = (int)((g.m + kTile - 1) / kTile), tiles_n = (int)((g.n + kTile - 1) / kTile);
  hipLaunchKernelGGL(gemm_f32_mfma, dim3((unsigned)(tiles_m * tiles_n * splits)), dim3(kThreads), 0, s,
                     static_cast<const float *>(g.a), static_cast<const float *>(g.b),
                     static_cast<float *>(g.c), g.m, g.n, g.k, g.lda, g.ldb, g.ldc, tiles_m,
                     tiles_n, splits, ws);
}

} // namespace vxk
