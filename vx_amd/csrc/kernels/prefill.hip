/*
 * prefill.hip -- the given positions of the int8 decoder (a prompt, a text
 * to score) as one pass over the weights for up to kPrefillCap of them,
 * where decode.hip's step reads every weight for each position.
 *
 * Same arithmetic as the step (the semantics of reference
 * examples/llama.vx:145-420): int8 weights with one f32 scale per row, f32
 * activations, f32 sums and softmax. Per layer, 7 launches:
 *
 *   prefill_norm             RMSNorm(x) as three bf16 planes
 *   prefill_gemm<kPreQkv>    [Wq; Wk; Wv], RoPE on q and k, k and v into the
 *                            cache
 *   prefill_attention        causal softmax(q k^T / sqrt(hs)) v, as planes
 *   prefill_gemm<kPreResid>  x += Wo att
 *   prefill_norm
 *   prefill_gemm<kPreSwiglu> [W1; W3] interleaved, silu(h1) * h3, as planes
 *   prefill_gemm<kPreResid>  x += W2 h
 *
 * The GEMMs run on bf16 MFMAs without giving up f32 activations: an f32
 * value is the exact sum of three bf16 values (its 24 significant bits, 8 at
 * a time, cut and not rounded, so that the first cannot overflow), an int8
 * weight is a bf16 value, and their products are exact in the f32 sums. The
 * first plane's sums and the other two's are kept apart and added at the
 * end, so the small terms' additions do not round the large sum.
 */
#include "../vx_hip_common.h"
#include "../vx_decode_kernels.h"
#include "vx_lds_dma.hip.h"
#include "vx_mfma16.hip.h"
#include "vx_wave_ops.hip.h"

#include <cmath>

namespace vxk {
namespace {

constexpr int kThreads = 256;

/* v = a + b + c exactly, each a bf16 value in the upper half of its word
 * (below 2^-110 the last bits of c are lost to bf16's smallest value, 2^-133).
 * An infinity or NaN goes into a alone. */
struct Split {
  uint32_t a, b, c;
};
__device__ __forceinline__ Split split3(float v) {
  const uint32_t u = __float_as_uint(v);
  const bool finite = (u & 0x7f800000u) != 0x7f800000u;
  Split s;
  s.a = u & 0xffff0000u;
  if (!finite && (u & 0x007fffffu)) {
    s.a |= 0x00400000u;
  }
  const float r = finite ? v - __uint_as_float(s.a) : 0.0f;
  s.b = __float_as_uint(r) & 0xffff0000u;
  s.c = __float_as_uint(r - __uint_as_float(s.b)) & 0xffff0000u;
  return s;
}

/* x[t] = the embedding row of tokens[t]. */
__global__ __launch_bounds__(kThreads) void prefill_embed(const int *tokens, const int8_t *tok_q,
                                                          const float *tok_s, float *x, int dim) {
  const int t = blockIdx.x;
  const int tok = tokens[t];
  const float s = tok_s[tok];
  const int8_t *row = tok_q + (int64_t)tok * dim;
  for (int i = threadIdx.x; i < dim; i += kThreads) {
    x[(int64_t)t * dim + i] = (float)row[i] * s;
  }
}

/* The planes of RMSNorm(x[t]) (reference examples/llama.vx:145-158). */
__global__ __launch_bounds__(kThreads) void prefill_norm(const float *__restrict__ x,
                                                         const float *__restrict__ w,
                                                         uint16_t *__restrict__ planes, int dim,
                                                         int kp) {
#pragma clang fp contract(off)
  __shared__ float part[kThreads / 64];
  const int64_t t = blockIdx.x;
  constexpr int kMost = kPrefillMaxCols / (4 * kThreads); /* float4 per thread */
  f32x4 v[kMost], nw[kMost];
  float ss = 0.0f;
#pragma unroll
  for (int k = 0; k < kMost; ++k) {
    const int i = 4 * (threadIdx.x + k * kThreads);
    if (i < dim) {
      v[k] = *reinterpret_cast<const f32x4 *>(x + t * dim + i);
      nw[k] = *reinterpret_cast<const f32x4 *>(w + i);
    }
  }
#pragma unroll
  for (int k = 0; k < kMost; ++k) {
    if (4 * (int)(threadIdx.x + k * kThreads) < dim) {
      ss += v[k][0] * v[k][0] + v[k][1] * v[k][1] + v[k][2] * v[k][2] + v[k][3] * v[k][3];
    }
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) {
    part[threadIdx.x >> 6] = ss;
  }
  __syncthreads();
  ss = 0.0f;
#pragma unroll
  for (int i = 0; i < kThreads / 64; ++i) {
    ss += part[i];
  }
  const float inv = 1.0f / sqrtf(ss / (float)dim + 0.00001f);
  const int64_t plane = (int64_t)kPrefillCap * kp;
#pragma unroll
  for (int k = 0; k < kMost; ++k) {
    const int i = 4 * (threadIdx.x + k * kThreads);
    if (i < dim) {
      Split s[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[e] = split3(nw[k][e] * (inv * v[k][e]));
      }
      uint16_t *dst = planes + t * kp + i;
      *reinterpret_cast<uint2 *>(dst) =
          uint2{(s[0].a >> 16) | s[1].a, (s[2].a >> 16) | s[3].a};
      *reinterpret_cast<uint2 *>(dst + plane) =
          uint2{(s[0].b >> 16) | s[1].b, (s[2].b >> 16) | s[3].b};
      *reinterpret_cast<uint2 *>(dst + 2 * plane) =
          uint2{(s[0].c >> 16) | s[1].c, (s[2].c >> 16) | s[3].c};
    }
  }
}

/* Eight int8 weights (two words) as four words of bf16 pairs. */
__device__ __forceinline__ u32x4 widen(uint32_t lo, uint32_t hi) {
  u32x4 r;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t w = h ? hi : lo;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const uint32_t f0 = __float_as_uint((float)(int8_t)(w >> (16 * e)));
      const uint32_t f1 = __float_as_uint((float)(int8_t)(w >> (16 * e + 8)));
      r[2 * h + e] = __builtin_amdgcn_perm(f1, f0, 0x07060302u); /* upper halves */
    }
  }
  return r;
}

enum PreMode { kPreQkv = 0, kPreResid = 1, kPreSwiglu = 2, kPreLogits = 3 };

/* out[t][r] = scale[r] * sum_k w[r][k] x[t][k] for kBT positions and kBR
 * rows a workgroup (4 waves, kWT of them along the positions), with the
 * mode's epilogue.
 *
 * K walks in stages of kKB through a kNS-slot LDS ring of buffer-to-LDS
 * loads, kNS - 1 stages ahead, one barrier a stage: the three planes of x and
 * the weight rows. A lane's 16 bytes of weights are k = 16 g .. 16 g + 15 of
 * a 64-block (g = lane / 16), used as two MFMA steps; the x operands follow
 * the same order of k. What bounds it is how long a stage's loads take to
 * arrive, so the ring is as deep as LDS allows.
 *
 * k past the row's end reads the next row's weights (zeros past the last)
 * against planes whose columns are zero up to kp; rows and positions past
 * the last compute what is not stored. */
template <int kMode, int kBT, int kBR, int kKB, int kWT, int kNS>
__global__ __launch_bounds__(kThreads, 1) void prefill_gemm(PrefillGemmArgs a) {
#pragma clang fp contract(off)
  constexpr int kNT = kBT / 16 / kWT;        /* 16-position blocks per wave */
  constexpr int kRB = kBR / 16 * kWT / 4;    /* 16-row blocks per wave */
  constexpr int kXC = kKB / 8;               /* 16-byte chunks of an x row */
  constexpr int kXUnits = 3 * kBT * kXC;     /* per stage */
  constexpr int kXL = kXUnits / kThreads;    /* loads per wave */
  constexpr int kWC = kKB / 16;              /* 16-byte chunks of a weight row */
  constexpr int kWUnits = kBR * kWC;
  constexpr int kWL = kWUnits / kThreads;
  static_assert(kXUnits % kThreads == 0 && kWUnits % kThreads == 0, "whole loads");
  __shared__ u32x4 ring[kNS][kXUnits + kWUnits];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15;
  const int g = lane >> 4;
  const int wr = wave / kWT * kRB * 16; /* the wave's first row in the tile */
  const int wt = wave % kWT * kNT * 16; /* and its first position */
  const int tok_tiles = (a.count + kBT - 1) / kBT;
  const int row0 = ((int)blockIdx.x / tok_tiles) * kBR;
  const int tok0 = ((int)blockIdx.x % tok_tiles) * kBT;
  const int K = a.cols;
  const int stages = (K + kKB - 1) / kKB;

  /* x: unit = (plane, position, chunk), chunk XORed with the position's low
   * bits so that 8 positions at one chunk are 8 distinct bank groups. */
  uint32_t x_off[kXL], w_off[kWL];
#pragma unroll
  for (int p = 0; p < kXL; ++p) {
    const int u = (wave * kXL + p) * 64 + lane;
    const int t = (u / kXC) % kBT, plane = u / (kXC * kBT);
    x_off[p] = (uint32_t)(((plane * kPrefillCap + t) * a.kp + ((u % kXC) ^ (t & 7)) * 8) * 2);
  }
  /* weights: unit = (row, chunk), swizzled likewise. */
  auto w_swz = [](int r, int c) {
    return kWC == 4 ? c ^ (((r >> 1) ^ (r >> 2)) & 3) : c ^ (r & 7);
  };
#pragma unroll
  for (int p = 0; p < kWL; ++p) {
    const int u = (wave * kWL + p) * 64 + lane;
    const int r = u / kWC;
    w_off[p] = (uint32_t)(r * K + w_swz(r, u % kWC) * 16);
  }
  const uint16_t *xb = a.x + (int64_t)tok0 * a.kp;
  const int x_bytes = (3 * kPrefillCap - tok0) * a.kp * 2;
  const int8_t *wb = a.w + (int64_t)row0 * K;
  /* the tile's rows; what lies past a range loads zeros */
  const int w_bytes = min(a.rows - row0, kBR) * K;
  const uint32_t ring_base = (uint32_t)(uintptr_t)(VX_LDS void *)&ring[0][0];
  auto issue = [&](int st, int slot) {
    const i32x4 rx = buffer_rsrc(xb + st * kKB, x_bytes - st * kKB * 2);
    const i32x4 rw = buffer_rsrc(wb + st * kKB, w_bytes - st * kKB);
    const uint32_t base = ring_base + (uint32_t)(slot * (kXUnits + kWUnits) * 16);
#pragma unroll
    for (int p = 0; p < kXL; ++p) {
      dma16(rx, x_off[p], base + (uint32_t)((wave * kXL + p) * 1024));
    }
#pragma unroll
    for (int p = 0; p < kWL; ++p) {
      dma16(rw, w_off[p], base + (uint32_t)((kXUnits + (wave * kWL + p) * 64) * 16));
    }
  };

  /* The epilogue's operands, requested before the first stage and there by
   * the last: row scales, the residual stream's old values, the rotary
   * factors. Lane: position l16 of each 16, rows 4 g .. 4 g + 3 of each 16,
   * as two pairs (rows are even, so a pair is whole or absent; an absent one
   * points past the range and loads zeros). */
  constexpr uint32_t kOut = 0x80000000u;
  const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(
      (void *)a.scale, (short)0, a.rows * 4, 0x00020000);
  u32x2 sc[kRB][2], ext[kMode == kPreQkv || kMode == kPreResid ? kRB : 1][kNT][2];
#pragma unroll
  for (int i = 0; i < kRB; ++i) {
    const int r = row0 + wr + i * 16 + 4 * g;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int r2 = r + 2 * h;
      sc[i][h] = __builtin_amdgcn_raw_buffer_load_b64(
          sr, (int)(r2 < a.rows ? (uint32_t)(r2 * 4) : kOut), 0, 0);
      if constexpr (kMode == kPreQkv) {
        const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(a.rope + (int64_t)a.pos0 * a.hs), (short)0, a.count * a.hs * 4, 0x00020000);
        const int c = r2 < a.dim ? r2 : r2 - a.dim;
#pragma unroll
        for (int j = 0; j < kNT; ++j) {
          const int t = tok0 + wt + j * 16 + l16;
          ext[i][j][h] = __builtin_amdgcn_raw_buffer_load_b64(
              rr, (int)(r2 < a.dim + a.kv_dim ? (uint32_t)((t * a.hs + c % a.hs) * 4) : kOut), 0, 0);
        }
      } else if constexpr (kMode == kPreResid) {
        const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
            (void *)a.out, (short)0, a.count * a.rows * 4, 0x00020000);
#pragma unroll
        for (int j = 0; j < kNT; ++j) {
          const int t = tok0 + wt + j * 16 + l16;
          ext[i][j][h] = __builtin_amdgcn_raw_buffer_load_b64(
              rr, (int)(r2 < a.rows ? (uint32_t)((t * a.rows + r2) * 4) : kOut), 0, 0);
        }
      }
    }
  }

  f32x4 hi[kRB][kNT], lo[kRB][kNT];
#pragma unroll
  for (int i = 0; i < kRB; ++i) {
#pragma unroll
    for (int j = 0; j < kNT; ++j) {
      hi[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      lo[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
#pragma unroll
  for (int s = 0; s < kNS - 1; ++s) {
    if (s < stages) {
      issue(s, s);
    }
  }
  for (int st = 0; st < stages; ++st) {
    wait_stages<kNS - 2, kXL + kWL>(min(stages - 1 - st, kNS - 2));
    lds_barrier();
    if (st + kNS - 1 < stages) {
      issue(st + kNS - 1, (st + kNS - 1) % kNS); /* the slot read last stage */
    }
    const u32x4 *xs = ring[st % kNS];
    const u32x4 *ws = xs + kXUnits;
#pragma unroll
    for (int b = 0; b < kKB / 64; ++b) {
      u32x4 wf[kRB][2];
#pragma unroll
      for (int i = 0; i < kRB; ++i) {
        const int r = wr + i * 16 + l16;
        const u32x4 q = ws[r * kWC + w_swz(r, 4 * b + g)];
        wf[i][0] = widen(q[0], q[1]);
        wf[i][1] = widen(q[2], q[3]);
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int j = 0; j < kNT; ++j) {
          const int t = wt + j * 16 + l16;
          const int c = (8 * b + 2 * g + s) ^ (t & 7);
          u32x4 xf[3];
#pragma unroll
          for (int p = 0; p < 3; ++p) {
            xf[p] = xs[(p * kBT + t) * kXC + c];
          }
#pragma unroll
          for (int i = 0; i < kRB; ++i) {
            hi[i][j] = mfma16<true>(wf[i][s], xf[0], hi[i][j]);
            lo[i][j] = mfma16<true>(wf[i][s], xf[1], lo[i][j]);
            lo[i][j] = mfma16<true>(wf[i][s], xf[2], lo[i][j]);
          }
        }
      }
    }
  }

#pragma unroll
  for (int j = 0; j < kNT; ++j) {
    const int t = tok0 + wt + j * 16 + l16;
    if (t >= a.count) {
      continue;
    }
#pragma unroll
    for (int i = 0; i < kRB; ++i) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int r2 = row0 + wr + i * 16 + 4 * g + 2 * h;
        if (r2 >= a.rows) {
          continue;
        }
        const float y0 =
            __uint_as_float(sc[i][h][0]) * (hi[i][j][2 * h] + lo[i][j][2 * h]);
        const float y1 =
            __uint_as_float(sc[i][h][1]) * (hi[i][j][2 * h + 1] + lo[i][j][2 * h + 1]);
        if constexpr (kMode == kPreQkv) {
          const int pos = a.pos0 + t;
          if (r2 < a.dim + a.kv_dim) {
            /* RoPE on the (even, odd) pair (reference :235-264). */
            const int c = r2 < a.dim ? r2 : r2 - a.dim;
            const float fr = __uint_as_float(ext[i][j][h][0]);
            const float fi = __uint_as_float(ext[i][j][h][1]);
            const float2 e{y0 * fr - y1 * fi, y0 * fi + y1 * fr};
            float *dst = r2 < a.dim ? a.out + (int64_t)t * a.dim + c
                                    : a.kcache + (int64_t)pos * a.kv_dim + c;
            *reinterpret_cast<float2 *>(dst) = e;
          } else {
            *reinterpret_cast<float2 *>(a.vcache + (int64_t)pos * a.kv_dim +
                                        (r2 - a.dim - a.kv_dim)) = float2{y0, y1};
          }
        } else if constexpr (kMode == kPreResid) {
          *reinterpret_cast<float2 *>(a.out + (int64_t)t * a.rows + r2) =
              float2{__uint_as_float(ext[i][j][h][0]) + y0,
                     __uint_as_float(ext[i][j][h][1]) + y1};
        } else if constexpr (kMode == kPreSwiglu) {
          /* rows 2i and 2i + 1 are W1's and W3's row i (reference :377-384). */
          const float neg = 0.0f - y0;
          float v = y0 * (1.0f / (1.0f + expf(neg)));
          v = v * y1;
          const Split s = split3(v);
          uint16_t *dst = a.planes + (int64_t)t * a.planes_kp + (r2 >> 1);
          const int64_t plane = (int64_t)kPrefillCap * a.planes_kp;
          dst[0] = (uint16_t)(s.a >> 16);
          dst[plane] = (uint16_t)(s.b >> 16);
          dst[2 * plane] = (uint16_t)(s.c >> 16);
        } else {
          *reinterpret_cast<float2 *>(a.out + (int64_t)t * a.rows + r2) = float2{y0, y1};
        }
      }
    }
  }
}

/* Max over the four lanes that share lane % 16. */
__device__ __forceinline__ float quad_rows_max(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}
__device__ __forceinline__ float quad_rows_sum(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

/* Causal attention of 16 query positions of one head (reference :275-325),
 * in f32 on v_mfma_f32_16x16x4_f32. The four waves take every fourth tile of
 * 16 keys straight from the cache into MFMA operands, each with its own
 * online softmax, and meet once in LDS. S^T = K Q^T leaves lane (query
 * l16, g) the scores of keys 4 g .. 4 g + 3, which is where O^T += V^T P^T
 * wants its B operand when k slot g of step r is key 4 g + r; Q and K operands
 * use float4 loads, with step e of slot g standing for d = 16 t + 4 g + e. */
template <int kHS> /* head size, or 16 for heads of up to 16 */
__global__ __launch_bounds__(kThreads) void prefill_attention(PrefillAttnArgs a) {
#pragma clang fp contract(off)
  constexpr int kDT = kHS / 16;
  __shared__ float so[4][16][kHS];
  __shared__ float sm[4][16], sl[4][16];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15;
  const int g = lane >> 4;
  const int hs = kHS == 16 ? a.hs : kHS;
  const int h = blockIdx.x;
  const int hk = h / a.kv_mul;
  const int q0 = blockIdx.y * 16;
  const int dim = (int)gridDim.x * hs;
  const int cache_bytes = a.seq_len * a.kv_dim * 4;
  const __amdgpu_buffer_rsrc_t krs =
      __builtin_amdgcn_make_buffer_rsrc((void *)a.kcache, (short)0, cache_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t vrs =
      __builtin_amdgcn_make_buffer_rsrc((void *)a.vcache, (short)0, cache_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t qrs = __builtin_amdgcn_make_buffer_rsrc(
      (void *)a.q, (short)0, a.count * dim * 4, 0x00020000);
  constexpr uint32_t kOut = 0x80000000u; /* past every range: zeros */

  /* Elements 16 t + 4 g .. + 3 of the head's row at byte `base`. */
  auto head4 = [&](__amdgpu_buffer_rsrc_t rs, uint32_t base, int t) -> f32x4 {
    const int d = 16 * t + 4 * g;
    if constexpr (kHS > 16) {
      return __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(base + 4 * d), 0, 0));
    } else {
      f32x4 r;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        r[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
            rs, (int)(d + e < hs ? base + 4 * (d + e) : kOut), 0, 0));
      }
      return r;
    }
  };
  f32x4 qf[kDT];
  const int qi = q0 + l16; /* this lane's query (zeros past the last) */
#pragma unroll
  for (int t = 0; t < kDT; ++t) {
    qf[t] = head4(qrs, qi < a.count ? (uint32_t)((qi * dim + h * hs) * 4) : kOut, t);
  }
  const int last = a.pos0 + qi; /* the last key this query sees */
  const int end = a.pos0 + min(q0 + 16, a.count); /* keys any query sees */
  auto load_k = [&](int k0, f32x4 (&kf)[kDT]) {
    const int key = k0 + l16;
    const uint32_t base = key < end ? (uint32_t)((key * a.kv_dim + hk * hs) * 4) : kOut;
#pragma unroll
    for (int t = 0; t < kDT; ++t) {
      kf[t] = head4(krs, base, t);
    }
  };
  auto load_v = [&](int k0, float (&vf)[4][kDT]) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int key = k0 + 4 * g + r;
#pragma unroll
      for (int t = 0; t < kDT; ++t) {
        const int d = 16 * t + l16;
        vf[r][t] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
            vrs, (int)(key < end && d < hs ? (uint32_t)((key * a.kv_dim + hk * hs + d) * 4) : kOut),
            0, 0));
      }
    }
  };

  const float root = sqrtf((float)hs);
  float m_run = -INFINITY, l_run = 0.0f;
  f32x4 o[kDT];
#pragma unroll
  for (int t = 0; t < kDT; ++t) {
    o[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  auto tile = [&](int k0, const f32x4 (&kf)[kDT], const float (&vf)[4][kDT]) {
    f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < kDT; ++t) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t][e], qf[t][e], s, 0, 0, 0);
      }
    }
    float mx = -INFINITY;
    float p[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      p[r] = k0 + 4 * g + r <= last ? s[r] / root : -INFINITY;
      mx = fmaxf(mx, p[r]);
    }
    mx = fmaxf(m_run, quad_rows_max(mx));
    const float m_use = mx == -INFINITY ? 0.0f : mx; /* no key seen yet */
    const float alpha = expf(m_run - m_use);
    float ps = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      p[r] = k0 + 4 * g + r <= last ? expf(p[r] - m_use) : 0.0f;
      ps = ps + p[r];
    }
    l_run = l_run * alpha + ps; /* this lane's keys; summed over g at the end */
    m_run = mx;
#pragma unroll
    for (int t = 0; t < kDT; ++t) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[t][e] = o[t][e] * alpha;
      }
    }
    /* A value past a query's last key must not reach it: 0 * Inf is NaN. Where
     * such a tile holds a value that is not finite, add key by key, each
     * where it is seen. */
    bool odd = false;
    if (k0 + 15 > a.pos0 + q0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int t = 0; t < kDT; ++t) {
          odd |= (__float_as_uint(vf[r][t]) & 0x7f800000u) == 0x7f800000u;
        }
      }
    }
    if (__builtin_amdgcn_ballot_w64(odd) == 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int t = 0; t < kDT; ++t) {
          o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[r][t], p[r], o[t], 0, 0, 0);
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        for (int kg = 0; kg < 4; ++kg) {
          const int key = k0 + 4 * kg + r;
          const float pk = __shfl(p[r], 16 * kg + l16);
#pragma unroll
          for (int t = 0; t < kDT; ++t) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float v = __shfl(vf[r][t], 16 * kg + 4 * g + e);
              o[t][e] = key <= last ? o[t][e] + pk * v : o[t][e];
            }
          }
        }
      }
    }
  };
  /* Two tiles in turn: the next one's loads go out before this one is used. */
  f32x4 k_a[kDT], k_b[kDT];
  float v_a[4][kDT], v_b[4][kDT];
  int k0 = wave * 16;
  if (k0 < end) {
    load_k(k0, k_a);
    load_v(k0, v_a);
  }
  for (; k0 < end; k0 += 128) {
    load_k(k0 + 64, k_b);
    load_v(k0 + 64, v_b);
    tile(k0, k_a, v_a);
    if (k0 + 64 >= end) {
      break;
    }
    load_k(k0 + 128, k_a);
    load_v(k0 + 128, v_a);
    tile(k0 + 64, k_b, v_b);
  }
  l_run = quad_rows_sum(l_run);
#pragma unroll
  for (int t = 0; t < kDT; ++t) {
    *reinterpret_cast<f32x4 *>(&so[wave][l16][16 * t + 4 * g]) = o[t];
  }
  if (g == 0) {
    sm[wave][l16] = m_run;
    sl[wave][l16] = l_run;
  }
  __syncthreads();
  const int q = threadIdx.x >> 4;
  if (q0 + q >= a.count) {
    return;
  }
  float mx = sm[0][q];
#pragma unroll
  for (int w = 1; w < 4; ++w) {
    mx = fmaxf(mx, sm[w][q]);
  }
  float f[4], den = 0.0f;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    f[w] = sm[w][q] == -INFINITY ? 0.0f : expf(sm[w][q] - mx);
    den = den + sl[w][q] * f[w];
  }
  const int64_t plane = (int64_t)kPrefillCap * a.kp;
#pragma unroll
  for (int t = 0; t < kDT; ++t) {
    const int d = 16 * t + (threadIdx.x & 15);
    if (d < hs) {
      float num = 0.0f;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        num = num + so[w][q][d] * f[w];
      }
      const Split s = split3(num / den);
      uint16_t *dst = a.planes + (int64_t)(q0 + q) * a.kp + h * hs + d;
      dst[0] = (uint16_t)(s.a >> 16);
      dst[plane] = (uint16_t)(s.b >> 16);
      dst[2 * plane] = (uint16_t)(s.c >> 16);
    }
  }
}

template <int kMode, int kBT, int kBR, int kKB, int kWT, int kNS>
void launch_gemm(const PrefillGemmArgs &a, hipStream_t s) {
  const int groups = ((a.rows + kBR - 1) / kBR) * ((a.count + kBT - 1) / kBT);
  hipLaunchKernelGGL((prefill_gemm<kMode, kBT, kBR, kKB, kWT, kNS>), dim3(groups), dim3(kThreads),
                     0, s, a);
}

/* Tile by grid. A layer's GEMM is a chain of stages whose loads must arrive,
 * so more workgroups with shorter stages beat larger tiles until every CU has
 * its share: 64 positions x 128 rows once there are two such tiles per CU (the
 * classifier), 64 x 64 once those fill the CUs, 32 x 64 once half of them are
 * busy, else 16 x 64. Prompt of 200 through the 12 layers of the dim-768
 * decoder and one classified position: 735 us so, 890 with 16 x 64 alone, 897
 * with 32 x 64, 966 with 64 x 64; prompt of 16: 547 so, 819 with 64 x 64. */
template <int kMode> void pick_gemm(const PrefillGemmArgs &a, hipStream_t s) {
  const int cus = device_cu_count();
  const int64_t r64 = (a.rows + 63) / 64;
  auto tiles = [&](int bt) { return (a.count + bt - 1) / bt; };
  if ((r64 + 1) / 2 * tiles(64) >= 2 * cus) {
    launch_gemm<kMode, 64, 128, 64, 2, 4>(a, s);
  } else if (a.count > 32 && r64 * tiles(64) >= cus) {
    launch_gemm<kMode, 64, 64, 64, 2, 5>(a, s);
  } else if (a.count > 16 && r64 * tiles(32) >= cus / 2) {
    launch_gemm<kMode, 32, 64, 64, 2, 8>(a, s);
  } else {
    launch_gemm<kMode, 16, 64, 128, 1, 7>(a, s);
  }
}

} // namespace

void prefill_embed_launch(const int *tokens, const int8_t *tok_q, const float *tok_s, float *x,
                          int count, int dim, hipStream_t s) {
  hipLaunchKernelGGL(prefill_embed, dim3(count), dim3(kThreads), 0, s, tokens, tok_q, tok_s, x, dim);
}

void prefill_norm_launch(const float *x, const float *w, uint16_t *planes, int count, int dim,
                         hipStream_t s) {
  hipLaunchKernelGGL(prefill_norm, dim3(count), dim3(kThreads), 0, s, x, w, planes, dim,
                     prefill_kp(dim));
}

void prefill_qkv_launch(const PrefillGemmArgs &a, hipStream_t s) { pick_gemm<kPreQkv>(a, s); }
void prefill_resid_launch(const PrefillGemmArgs &a, hipStream_t s) { pick_gemm<kPreResid>(a, s); }
void prefill_swiglu_launch(const PrefillGemmArgs &a, hipStream_t s) { pick_gemm<kPreSwiglu>(a, s); }
void prefill_logits_launch(const PrefillGemmArgs &a, hipStream_t s) { pick_gemm<kPreLogits>(a, s); }

void prefill_attention_launch(const PrefillAttnArgs &a, int heads, hipStream_t s) {
  const dim3 grid(heads, (a.count + 15) / 16);
  switch (a.hs) {
  case 32: hipLaunchKernelGGL((prefill_attention<32>), grid, dim3(kThreads), 0, s, a); break;
  case 64: hipLaunchKernelGGL((prefill_attention<64>), grid, dim3(kThreads), 0, s, a); break;
  case 128: hipLaunchKernelGGL((prefill_attention<128>), grid, dim3(kThreads), 0, s, a); break;
  case 256: hipLaunchKernelGGL((prefill_attention<256>), grid, dim3(kThreads), 0, s, a); break;
  default: hipLaunchKernelGGL((prefill_attention<16>), grid, dim3(kThreads), 0, s, a); break;
  }
}

} // namespace vxk
