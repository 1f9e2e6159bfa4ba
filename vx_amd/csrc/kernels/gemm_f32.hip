/*
 * gemm_f32.hip -- f32 GEMM for products large enough that the exact-order
 * kernel's rate matters, on bf16 MFMAs, or on f32 MFMAs where K is short.
 *
 * An f32 value is the exact sum of three bf16 values, each the rest of the one
 * before rounded to nearest, and the product of two such values is exact in
 * f32. Of the nine products of a pair the six largest are added: the first in
 * one accumulator, the other five in a second, added at the end. The rounded
 * rests are at most 2^-8 and 2^-17 of the value's leading bit, so that what is
 * left out is at most 2^-24 of the product, of either sign.
 * Six v_mfma_f32_16x16x32_bf16 do 32 of k in 96 cycles; f32 MFMAs take 256.
 *
 * What bf16 cannot hold is left to f32 MFMAs: a block of 16 x 16 sums is
 * computed again that way, over the workgroup's k, where one of them is not
 * finite or lies below 2^-100 (but not 0), or where an element below 2^-100 may have lost
 * bits that count in it. The last needs, of each row and column, the greatest
 * magnitude and whether it has such an element; a tile that met one reads its
 * operands again for them (2048^3 with a third of A below 2^-110 124 us, with
 * an infinity in every tile 154, against 248 where all is done in f32).
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
 * K below f32::kPlanesMinK: the same tile on f32 MFMAs throughout, stages of 16
 * through one LDS slot and three workgroups to a CU, whose loads and stores
 * overlap. Writing C bounds it. The planes' way there, against it: 8192^2 x 16
 * 103 us, 47; 64280 x 2576 x 18 247, 148; 4096^2 x 64 34, 30; 8 x 8388608 x 16
 * 1195, 500. (Stages of 32: 52, 168, 29 and 590; four workgroups to a CU spill:
 * 49, 162, 29 and 482.)
 *
 * Against f32 MFMAs in the same tile: 2048^3 248 -> 90 us with new inputs each
 * pass (191 TFLOP/s); error against 64 bits 8.1e-7 -> 2.5e-7 at 2048^3, 1.1e-6
 * -> 3.8e-7 at K = 4096. Watching the least magnitude is 3% of that (24 of a
 * stage's 120 vector instructions a wave). Grids of fewer tiles than CUs divide
 * K over workgroups: 1024^3 125 -> 25 us (undivided 45), 128 x 4096 x 4096 454
 * -> 37 (142).
 */
#include "../vx_hip_common.h"
#include "../vx_kernels.h"
#include "gemm_f32.h"
#include "gemm_pp_layout.h"
#include "vx_lds_dma.hip.h"
#include "vx_mfma16.hip.h"
#include "vx_wave_ops.hip.h"

namespace vxk {
namespace {

constexpr int kThreads = 512;
constexpr int kTile = f32::kTile;
constexpr int kPlane = kTile * 4;     /* 16-byte units */
constexpr float kLeast = 7.888609052210118e-31f; /* 2^-100 */
constexpr uint32_t kLeastBits = (127 - 100) << 23;

struct __attribute__((packed, aligned(4))) Four {
  f32x4 v;
};

/* A thread's k of a stage: of one row of A and of one column of B. */
template <int kPer> struct Regs {
  float a[kPer], b[kPer];
};

__device__ __forceinline__ int unit(int row, int c) { return row * 4 + (c ^ ((row >> 1) & 3)); }
/* The same in f32, a chunk being 4 k, kC of them a row. */
template <int kC> __device__ __forceinline__ int unit32(int row, int c) {
  return kC == 4 ? unit(row, c) : row * kC + (c ^ (row & (kC - 1)));
}

/* Two values rounded to bf16, the first in the lower half. */
__device__ __forceinline__ uint32_t round2(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), bf16x2));
}

/* Eight values as the three planes' 16 bytes. */
__device__ __forceinline__ void split8(const float (&x)[8], u32x4 (&p)[3]) {
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    float lo = x[2 * w], hi = x[2 * w + 1];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const uint32_t r = round2(lo, hi);
      p[i][w] = r;
      lo -= __uint_as_float(r << 16);
      hi -= __uint_as_float(r & 0xffff0000u);
    }
  }
}

template <bool kPlanes>
__global__ __launch_bounds__(kThreads, kPlanes ? 2 : 7) void gemm_f32_mfma(
    const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ C, int64_t M,
    int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int tiles_m, int tiles_n,
    int splits, char *__restrict__ ws) {
  constexpr int kPer = kPlanes ? 8 : 4;  /* of k per thread and stage */
  constexpr int kKs = 4 * kPer;
  constexpr int kC = kKs / 4;            /* chunks of a row in f32 */
  constexpr int kRows32 = kTile * kC;    /* 16-byte units of a stage's rows in f32 */
  using Regs = vxk::Regs<kPer>;
  /* [slot][A, B][plane][kPlane]; in f32 [slot][A, B][kRows32], one slot alone */
  __shared__ u32x4 lds[kPlanes ? 2 * 2 * 3 * kPlane : 2 * kRows32];
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
  const float *pa = A + min(m0 + a_row, M - 1) * lda + first * kKs + kPer * a_chunk;
  const int b_off = (int)(min(n0 + b_col, N - 1) - n0);
  const float *pb = B + (first * kKs + kPer * b_chunk) * ldb + n0;

  auto load = [&](Regs &r, int64_t st) {
    const float *a = pa + st * kKs;
    const float *b = pb + st * kKs * ldb;
#pragma unroll
    for (int h = 0; h < kPer / 4; ++h) {
      const f32x4 v = reinterpret_cast<const Four *>(a)[h].v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        r.a[4 * h + e] = v[e];
      }
    }
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
      r.b[e] = (b + e * ldb)[b_off];
    }
  };
  auto load_last = [&](Regs &r, int64_t st) { /* zeros past K */
    const float *a = pa + st * kKs;
    const float *b = pb + st * kKs * ldb;
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
      r.a[e] = st * kKs + kPer * a_chunk + e < left ? a[e] : 0.0f;
      r.b[e] = st * kKs + kPer * b_chunk + e < left ? (b + e * ldb)[b_off] : 0.0f;
    }
  };
  auto load_any = [&](Regs &r, int64_t st) {
    if (st < whole) {
      load(r, st);
    } else {
      load_last(r, st);
    }
  };

  /* c[i][j]: rows 64 wm + 16 i + l16, columns 32 wn + 16 j + 4 g .. + 3 */
  f32x4 c[4][2];

  /* The blocks of c whose bit 2 i + j is set, over the workgroup's k, on
   * v_mfma_f32_16x16x4_f32. Step e of a 16-k half takes k = 4 g + e of it from
   * lane group g, on both sides, so an operand is four steps' 16 bytes. */
  auto in_f32 = [&](uint32_t blocks) {
    auto stash = [&](const Regs &r, int slot) {
#pragma unroll
      for (int h = 0; h < kPer / 4; ++h) {
        lds[2 * slot * kRows32 + unit32<kC>(a_row, kPer / 4 * a_chunk + h)] = __builtin_bit_cast(
            u32x4, f32x4{r.a[4 * h], r.a[4 * h + 1], r.a[4 * h + 2], r.a[4 * h + 3]});
        lds[(2 * slot + 1) * kRows32 + unit32<kC>(b_col, kPer / 4 * b_chunk + h)] = __builtin_bit_cast(
            u32x4, f32x4{r.b[4 * h], r.b[4 * h + 1], r.b[4 * h + 2], r.b[4 * h + 3]});
      }
    };
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      if (blocks >> q & 1) {
        c[q >> 1][q & 1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      }
    }
    Regs r;
    load_any(r, 0);
    if constexpr (kPlanes) {
      stash(r, 0);
      if (stages > 1) {
        load_any(r, 1);
      }
      lds_barrier();
    }
    for (int64_t st = 0; st < stages; ++st) {
      const int slot = kPlanes ? (int)(st & 1) : 0;
      if constexpr (kPlanes) {
        if (st + 1 < stages) {
          stash(r, slot ^ 1);
        }
        if (st + 2 < stages) {
          load_any(r, st + 2);
        }
      } else {
        stash(r, 0);
        if (st + 1 < stages) {
          load_any(r, st + 1);
        }
        lds_barrier();
      }
#pragma unroll
      for (int h = 0; h < kC / 4; ++h) {
        if (st * kKs + 16 * h < left) {
          f32x4 af[4], bf[2];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            af[i] = __builtin_bit_cast(
                f32x4, lds[2 * slot * kRows32 + unit32<kC>(64 * wm + 16 * i + l16, 4 * h + g)]);
          }
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            bf[j] = __builtin_bit_cast(
                f32x4, lds[(2 * slot + 1) * kRows32 + unit32<kC>(32 * wn + 16 * j + l16, 4 * h + g)]);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              if (!kPlanes || (blocks >> (2 * i + j) & 1)) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  c[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[j][e], af[i][e], c[i][j], 0, 0, 0);
                }
              }
            }
          }
        }
      }
      lds_barrier();
    }
  };

  if constexpr (!kPlanes) {
    in_f32(~0u);
  } else {
    __shared__ int again;
    if (t == 0) {
      again = 0;
    }
    /* The least magnitude but zero, as its bits times two, less one. */
    constexpr uint32_t kTiny = 2 * kLeastBits - 1;
    uint32_t least = ~0u;
    auto stash = [&](const Regs &r, int slot) {
      u32x4 p[3];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        least = min(least, 2 * __float_as_uint(r.a[e]) - 1);
        least = min(least, 2 * __float_as_uint(r.b[e]) - 1);
      }
      split8(r.a, p);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        lds[(6 * slot + i) * kPlane + unit(a_row, a_chunk)] = p[i];
      }
      split8(r.b, p);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        lds[(6 * slot + 3 + i) * kPlane + unit(b_col, b_chunk)] = p[i];
      }
    };
    f32x4 lo[4][2];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      c[q >> 1][q & 1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      lo[q >> 1][q & 1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    u32x4 af[3][4], bf[3][2];
    auto fragments = [&](int slot) {
#pragma unroll
      for (int p = 0; p < 3; ++p) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          bf[p][j] = lds[(6 * slot + 3 + p) * kPlane + unit(32 * wn + 16 * j + l16, g)];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          af[p][i] = lds[(6 * slot + p) * kPlane + unit(64 * wm + 16 * i + l16, g)];
        }
      }
    };
    auto multiply = [&]() {
      auto add = [&](int pa_, int pb_, f32x4 (&x)[4][2]) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            x[i][j] = mfma16<true>(bf[pb_][j], af[pa_][i], x[i][j]);
          }
        }
      };
      add(0, 0, c);
      add(0, 1, lo);
      add(1, 0, lo);
      add(1, 1, lo);
      add(0, 2, lo);
      add(2, 0, lo);
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
        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0); /* VALU */
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

    uint32_t small = least, large = 0; /* of the sums, likewise, and the greatest */
#pragma unroll
    for (int q = 0; q < 8; ++q) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = c[q >> 1][q & 1][e] + lo[q >> 1][q & 1][e];
        c[q >> 1][q & 1][e] = v;
        small = min(small, 2 * __float_as_uint(v) - 1);
        large = max(large, __float_as_uint(v) & 0x7fffffffu);
      }
    }
    if (small < kTiny || large >= 0x7f800000u) {
      again = 1;
    }
    __syncthreads();
    if (again) {
      /* Blocks of c to compute again (bit 2 i + j): sums that are not finite,
       * or too small for the planes' products. */
      uint32_t odd = 0;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = __builtin_fabsf(c[q >> 1][q & 1][e]);
          odd |= (uint32_t)(!(v < INFINITY) || (v > 0.0f && v < kLeast)) << q;
        }
      }
      if (__syncthreads_or(least < kTiny)) {
        /* What such values may have lost, at most 2^-126 of each, against the
         * result: the rows' and columns' greatest and least are read again. */
        float a_max = 0.0f, b_max = 0.0f;
        uint32_t a_min = ~0u, b_min = ~0u;
        for (st = 0; st < stages; st += 3) {
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            load_any(r[i], min(st + i, stages - 1));
          }
#pragma unroll
          for (int i = 0; i < 3; ++i) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              a_max = fmaxf(a_max, __builtin_fabsf(r[i].a[e]));
              b_max = fmaxf(b_max, __builtin_fabsf(r[i].b[e]));
              a_min = min(a_min, 2 * __float_as_uint(r[i].a[e]) - 1);
              b_min = min(b_min, 2 * __float_as_uint(r[i].b[e]) - 1);
            }
          }
        }
        struct Side {
          float most, tiny; /* `tiny`: whether there is one, 1 or 0 */
        };
        Side *rows = reinterpret_cast<Side *>(&lds[0]); /* [4][128] each */
        Side *cols = rows + 4 * kTile;
        rows[a_chunk * kTile + a_row] = Side{a_max, a_min < kTiny ? 1.0f : 0.0f};
        cols[b_chunk * kTile + b_col] = Side{b_max, b_min < kTiny ? 1.0f : 0.0f};
        __syncthreads();
        auto side = [&](const Side *of, int at) {
          Side x = of[at];
#pragma unroll
          for (int q = 1; q < 4; ++q) {
            x.most = fmaxf(x.most, of[q * kTile + at].most);
            x.tiny = fmaxf(x.tiny, of[q * kTile + at].tiny);
          }
          return x;
        };
        const float lost = (float)(stages * kKs) * (kLeast * 2.0f);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const Side b = side(cols, 32 * wn + 16 * j + 4 * g + e);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const Side a = side(rows, 64 * wm + 16 * i + l16);
              odd |= (uint32_t)(lost * (a.tiny * b.most + b.tiny * a.most) >
                                __builtin_fabsf(c[i][j][e]))
                     << (2 * i + j);
            }
          }
        }
      }
      uint32_t blocks = 0; /* of the wave */
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        blocks |= (uint32_t)(__builtin_amdgcn_ballot_w64((odd >> q & 1) != 0) != 0) << q;
      }
      if (__syncthreads_or(blocks != 0)) {
        in_f32(blocks);
      }
    }
  }

  if (splits > 1) {
    /* The sums go past the caches that other XCDs do not see; the workgroup
     * with the last ticket adds all of them up in order. */
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(ws + split::kTicketBytes + (int64_t)id * splits * f32::kPart), (short)0,
        splits * f32::kPart, 0x00020000);
    const int at = t * 16;
    __shared__ int last;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, c[i][j]), wr,
                                               at + (2 * i + j) * kThreads * 16,
                                               split * f32::kPart, 16 /* sc1 */);
      }
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
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          c[i][j] = s == 0 ? v[i][j] : c[i][j] + v[i][j];
        }
      }
    }
  }
  /* Lanes of rows 2 r and 2 r + 1 trade a block, so that a store has whole
   * 128-byte lines: eight rows of 32 columns. */
  const int64_t col = n0 + 32 * wn + 16 * (l16 & 1) + 4 * g;
  auto store = [&](int64_t row, f32x4 v) {
    if (row < M && col < N) {
      float *p = C + row * ldc + col;
      if (col + 3 < N) {
        reinterpret_cast<Four *>(p)->v = v;
      } else {
#pragma unroll
        for (int e = 0; e < 3; ++e) {
          if (col + e < N) {
            p[e] = v[e];
          }
        }
      }
    }
  };
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f32x4 v0, v1;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float other = partner<1>((l16 & 1) ? c[i][0][e] : c[i][1][e]);
      v0[e] = (l16 & 1) ? other : c[i][0][e];
      v1[e] = (l16 & 1) ? c[i][1][e] : other;
    }
    const int64_t row = m0 + 64 * wm + 16 * i + (l16 & ~1);
    store(row, v0);
    store(row + 1, v1);
  }
}

} // namespace

void gemm_f32_launch(const GemmArgs &g, int splits, char *ws, hipStream_t s) {
  const int tiles_m = (int)((g.m + kTile - 1) / kTile), tiles_n = (int)((g.n + kTile - 1) / kTile);
  const auto kernel = g.k < f32::kPlanesMinK ? gemm_f32_mfma<false> : gemm_f32_mfma<true>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles_m * tiles_n * splits)), dim3(kThreads), 0, s,
                     static_cast<const float *>(g.a), static_cast<const float *>(g.b),
                     static_cast<float *>(g.c), g.m, g.n, g.k, g.lda, g.ldb, g.ldc, tiles_m,
                     tiles_n, splits, ws);
}

} // namespace vxk
