// Chunk GEMM tiles that dequantise int4-hier weights in registers:
// y[j] (+)= W x[j] + b over rows of 128-column steps, the last whole or half
// (in_f % 64 == 0, at least 128).
// reference: chunk_gemm.cu:65-176.
//
// * A lane's MFMA operand (v_mfma_f32_32x32x16_f16: row lane % 32, eight
//   consecutive k of the half lane / 32) is one packed word of a weight row,
//   so the weights go from memory to the matrix cores through registers only:
//   no LDS round trip and no barrier for them. A lane owns whole groups (one
//   16-byte load each): half h of a 128-column step has groups h and 2 + h,
//   and the k positions of an MFMA stand for word j of those two groups. x is
//   read from LDS at the same columns.
// * Dequantisation is w = f16(q * s + m) in one v_fma_mix per weight: the
//   nibble, masked in place, is an f16 subnormal q * 2^-24 (or q * 2^-20, the
//   odd nibbles), and s carries the 2^24. q * s is exact in f32 (11 + 4 + 4
//   bits), so the weight is rounded once, to f16. 13 VALU ops a word (5 of
//   ~2.6 clk, 8 of ~9 clk); the convert-fma-convert form it replaces took 36.
// * x goes memory -> LDS by DMA (global_load_lds_dwordx4), one step ahead, in
//   two buffers; a token's 16-byte chunk c sits at slot c ^ (token % 16), so
//   the 16 lanes of a read phase touch all 64 banks once. One barrier a step.
// * Inside a step the next MFMA's operands are read and dequantised under the
//   current MFMAs (sched_group_barrier).
// * x is the MFMA's row operand: a lane's accumulators hold 16 tokens of one
//   weight row, so a store instruction writes whole 128-byte row pieces and
//   needs no pass through LDS; a gate row and its up row (and a RoPE pair) sit
//   in one lane.
// * F16 weights (wst_gemm_fp16) run the same loop with the operand loaded as it
//   is: 896 -> 151936 x 256 tokens 292 -> 173 us (each load instruction touches
//   32 rows, which bounds it: the f16 products stay far from the matrix cores'
//   rate).
// * Every shape sums k in the same order, so a token's bits do not depend on
//   the tile, only on the K split.
//
// Measured, 0.5B gate|up + SwiGLU over 4096 tokens: 129-152 us on the 64 x 256
// LDS tiles, 84 us here (850 TFLOP/s); 7B gate|up over 4096 tokens 1,586 ->
// 1,090 us (1,020 TFLOP/s; an f16 library product of that size, weights
// already f16, reaches about 1,200: the chip's power limit on such data).
#pragma once
#include "common.hpp"

typedef _Float16 gt_h8 __attribute__((ext_vector_type(8)));
typedef _Float16 gt_h2 __attribute__((ext_vector_type(2)));
typedef float gt_f16v __attribute__((ext_vector_type(16)));
typedef uint32_t gt_u4 __attribute__((ext_vector_type(4)));

typedef uint32_t gt_u32a2 __attribute__((aligned(2)));

#define GT_KC 128           // columns per step: four int4-hier groups
// VALU ops scheduled after each MFMA: a k-step's dequantisations over its MFMAs
#define GT_VPM (F16 ? 1 : (13 * MT + MT * NT - 1) / (MT * NT) + 1)
#define GT_XROW (GT_KC * 2) // bytes of a token's step in LDS

struct GtRope {
  uint16_t *k_cache, *v_cache;
  const float *cos_tab, *sin_tab;
  const uint16_t *q_norm_w, *k_norm_w;
  int n_q, n_kv, pos0, max_seq;
  float eps;
};

// GT_ROPE64 / GT_ROPE128: the qkv projection's RoPE epilogue for that head size.
enum { GT_PLAIN = 0, GT_SWIGLU = 1, GT_ROPE64 = 2, GT_ROPE128 = 3 };

template <int WM_, int WN_, int MT_, int NT_>
struct GtShape {
  static constexpr int WM = WM_, WN = WN_, MT = MT_, NT = NT_;
  static constexpr int WAVES = WM * WN, THREADS = 64 * WAVES;
  static constexpr int BM = WM * MT * 32, BN = WN * NT * 32;
  static constexpr int XBUF = BN * GT_XROW;
  static constexpr int LDS = 2 * XBUF;
  static constexpr int XDMA = BN / (4 * WAVES);  // 1 KB DMA ops a wave issues per step
  static_assert(BN % (4 * WAVES) == 0, "whole DMA ops per wave");
  static_assert(LDS <= 160 * 1024, "one CU's LDS");
};

// Eight weights of one packed word as an MFMA operand.
__device__ __forceinline__ gt_h8 gt_dequant(uint32_t w, float s, float s16, float m) {
  const uint32_t u = w >> 8;
  const gt_h2 t0 = __builtin_bit_cast(gt_h2, w & 0x000F000Fu);
  const gt_h2 t1 = __builtin_bit_cast(gt_h2, w & 0x00F000F0u);
  const gt_h2 t2 = __builtin_bit_cast(gt_h2, u & 0x000F000Fu);
  const gt_h2 t3 = __builtin_bit_cast(gt_h2, u & 0x00F000F0u);
  gt_h8 r;
  r[0] = (_Float16)__builtin_fmaf((float)t0[0], s, m);
  r[1] = (_Float16)__builtin_fmaf((float)t1[0], s16, m);
  r[2] = (_Float16)__builtin_fmaf((float)t2[0], s, m);
  r[3] = (_Float16)__builtin_fmaf((float)t3[0], s16, m);
  r[4] = (_Float16)__builtin_fmaf((float)t0[1], s, m);
  r[5] = (_Float16)__builtin_fmaf((float)t1[1], s16, m);
  r[6] = (_Float16)__builtin_fmaf((float)t2[1], s, m);
  r[7] = (_Float16)__builtin_fmaf((float)t3[1], s16, m);
  return r;
}

template <int MT, bool F16>
struct GtW {
  // int4: groups half and 2 + half of the step; f16: the eight k-steps' operands
  gt_u4 q[MT][F16 ? 8 : 2];
  uint32_t ix[MT];  // int4: the step's four index bytes
};

// qw/si/sb: the weights [rows][in_f] (rows = out_f, or 2 out_f for the SwiGLU
// form); split blockIdx.y covers steps [y sps, min(steps, (y + 1) sps)) and
// writes ws[y] when ws is given. nb token tiles, `tiles` tiles; rfast: row
// tiles vary fastest. 32-bit offsets: n in_f 2, rows in_f / 2 and n out_f 4
// are below 2^31 (the host checks).
// TAIL: rows end in half a step (in_f % 128 == 64): the last step has groups 0
// and 1 only and skips the other four of its eight k-steps.
// F16: w is f16 [rows][in_f] (si and sb unused): a lane's operand is 16 bytes of
// a row, loaded straight into registers; k-step i covers columns 16 i .. 16 i +
// 15.
template <class S, int EPI, bool TAIL, bool F16>
__global__ __launch_bounds__(S::THREADS, S::MT * S::NT > 8 ? 1 : 2) void gemm_tile_kernel(
    const void *__restrict__ qw, const uint8_t *__restrict__ si, const uint32_t *__restrict__ sb,
    const uint16_t *__restrict__ x, const uint16_t *__restrict__ bias, float *__restrict__ y,
    float *__restrict__ ws, int in_f, int out_f, int n, int accum, int nb, int tiles, int sps, int rfast,
    GtRope re) {
  constexpr int MT = S::MT, NT = S::NT;
  extern __shared__ __align__(16) unsigned char gt_lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % S::WM, wn = wave / S::WM;
  const int l32 = lane & 31, half = lane >> 5;

  // XCD-aware order: blocks b, b + 8, ... share an XCD; give each XCD a
  // contiguous run of tiles, token tiles fastest (they share W rows).
  int b = blockIdx.x;
  {
    const int per = tiles >> 3, rem = tiles & 7;
    const int xcd = b & 7, loc = b >> 3;
    b = xcd * per + min(xcd, rem) + loc;
  }
  const int mb = tiles / nb;
  const int tm = rfast ? b % mb : b / nb, tn = rfast ? b / mb : b % nb;
  const int t0 = tn * S::BN;
  const int G = in_f >> 5;
  const int whole = in_f / GT_KC;  // whole steps of a row
  const int step0 = blockIdx.y * sps, step1 = min(whole + (TAIL ? 1 : 0), step0 + sps);

  uint32_t woff[MT], ioff[MT];
  float ds[MT], dm[MT];
#pragma unroll
  for (int f = 0; f < MT; ++f) {
    int r;
    if constexpr (EPI == GT_SWIGLU) {
      // Two fragments a wave: a gate row and its up row in one lane. One
      // fragment: the lower half of the waves takes gate rows, the upper half
      // their up rows.
      static_assert(EPI != GT_SWIGLU || MT == 2 || (MT == 1 && S::WM % 2 == 0), "gate and up");
      const int g = MT == 2 ? wm : wm % (S::WM / 2);
      r = min(tm * (S::BM / 2) + g * 32 + l32, out_f - 1) +
          ((MT == 2 ? f : wm / (S::WM / 2)) ? out_f : 0);
    } else if constexpr (EPI == GT_ROPE128) {
      // heads of 128 rows, two waves each: a wave has columns j and j + 64
      r = min(tm * S::BM + (wm >> 1) * 128 + f * 64 + (wm & 1) * 32 + l32, out_f - 1);
    } else {
      r = min(tm * S::BM + (wm * MT + f) * 32 + l32, out_f - 1);
    }
    if constexpr (F16) {
      ds[f] = dm[f] = 0.0f;
      woff[f] = (uint32_t)r * (uint32_t)(in_f * 2) + (uint32_t)half * 16u;
      ioff[f] = 0;
    } else {
      const uint32_t p = sb[r];
      ds[f] = h2f((uint16_t)(p & 0xFFFFu)) * 16777216.0f;
      dm[f] = -h2f((uint16_t)(p >> 16));
      woff[f] = (uint32_t)r * (uint32_t)(in_f / 2) + (uint32_t)half * 16u;
      ioff[f] = (uint32_t)r * (uint32_t)G;
    }
  }
  uint32_t xoff[S::XDMA];
#pragma unroll
  for (int i = 0; i < S::XDMA; ++i) {
    const int tl = (wave * S::XDMA + i) * 4 + (lane >> 4);
    const int tok = min(t0 + tl, n - 1);
    xoff[i] = (uint32_t)tok * (uint32_t)in_f * 2u + (uint32_t)(((lane & 15) ^ (tl & 15)) * 16);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)gt_lds;

  // A tail step's second half re-reads its first (nothing past a row is read).
  auto load_x = [&](int st, int buf) {
    const uint16_t *xs = x + (size_t)st * GT_KC;
    const bool tail = TAIL && st == whole;
    const uint32_t dst = lds0 + (uint32_t)buf * S::XBUF + (uint32_t)wave * (S::XDMA * 1024u);
#pragma unroll
    for (int i = 0; i < S::XDMA; ++i) {
      uint32_t off = xoff[i];
      if constexpr (TAIL) {
        const int tl = (wave * S::XDMA + i) * 4 + (lane >> 4);
        off -= tail ? (uint32_t)((lane ^ tl) & 8) * 16u : 0u;  // chunk 8 and on: chunk - 8
      }
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                   ::"s"(dst + i * 1024u), "v"(off), "s"(xs)
                   : "memory");
    }
  };
  auto load_w = [&](int st, GtW<MT, F16> &w) {
    const bool tail = TAIL && st == whole;
    if constexpr (F16) {
      const char *ws_ = (const char *)qw + (size_t)st * (GT_KC * 2);
#pragma unroll
      for (int f = 0; f < MT; ++f)
#pragma unroll
        for (int i = 0; i < 8; ++i)
          w.q[f][i] = *(const gt_u4 *)(ws_ + woff[f] + (tail && i >= 4 ? i - 4 : i) * 32u);
      return;
    }
    const char *qs = (const char *)qw + (size_t)st * (GT_KC / 2);
    // index bytes: a tail's two are the upper half of the word that ends with
    // the row (rows of an odd number of group pairs are 2-byte aligned)
    const uint8_t *is = si + (size_t)st * 4 - (tail ? 2 : 0);
#pragma unroll
    for (int f = 0; f < MT; ++f) {
      w.q[f][0] = *(const gt_u4 *)(qs + woff[f]);
      w.q[f][1] = *(const gt_u4 *)(qs + woff[f] + (tail ? 0u : 32u));
      if constexpr (TAIL)
        w.ix[f] = *(const gt_u32a2 *)(is + ioff[f]);
      else
        w.ix[f] = *(const uint32_t *)(is + ioff[f]);
    }
  };
  gt_f16v acc[MT][NT];
#pragma unroll
  for (int f = 0; f < MT; ++f)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[f][t][r] = 0.0f;

  // token wn * NT * 32 + 32 t + l32, chunk c at slot c ^ (token % 16)
  const uint32_t xbase = (uint32_t)((wn * NT * 32 + l32) * GT_XROW);
  const uint32_t xsw = (uint32_t)((F16 ? half : 4 * half) ^ (l32 & 15)) << 4;
  // The step's eight MFMA k-steps i (groups 2 (i / 4) + half, word i % 4):
  // the next k-step's operands are read and dequantised under this one's
  // MFMAs.
  // A tail step's index bytes sit in the upper half of the word, and its last
  // four k-steps are left out: nothing past a row's end is multiplied (zeros in
  // their place would make NaN of an infinite x or scale).
  auto compute = [&](const GtW<MT, F16> &w, int buf, int st) {
    const int sh = 8 * half + (TAIL && st == whole ? 16 : 0);
    const unsigned char *xb = gt_lds + buf * S::XBUF + xbase;
    gt_h8 xf[2][NT], wf[2][MT];
    float sc[MT], sc16[MT], mm[MT];
    auto scales = [&](int s) {
      if constexpr (F16) return;
#pragma unroll
      for (int f = 0; f < MT; ++f) {
        const uint32_t ix = (w.ix[f] >> sh) >> (16 * s);
        sc[f] = ds[f] * (float)(ix & 0xFu);
        sc16[f] = sc[f] * 0.0625f;
        mm[f] = dm[f] * (float)((ix >> 4) & 0xFu);
      }
    };
    auto read_x = [&](int i) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        xf[i & 1][t] = *(const gt_h8 *)(xb + t * 32 * GT_XROW +
                                        (xsw ^ (uint32_t)((F16 ? 2 * i : 8 * (i >> 2) + (i & 3)) * 16)));
      }
    };
    auto make_w = [&](int i) {
#pragma unroll
      for (int f = 0; f < MT; ++f) {
        if constexpr (F16)
          wf[i & 1][f] = __builtin_bit_cast(gt_h8, w.q[f][i]);
        else
          wf[i & 1][f] = gt_dequant(w.q[f][i >> 2][i & 3], sc[f], sc16[f], mm[f]);
      }
    };
    scales(0);
    read_x(0);
    make_w(0);
    __builtin_amdgcn_sched_barrier(0);
    // The multiplying wave goes first on its SIMD (with several blocks a CU:
    // 3584 -> 37888 x 5 tokens 30.6 -> 26.1 us, 18944 -> 3584 x 10 14.5 -> 13.1).
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (TAIL && i == 4 && st == whole) break;  // (uniform)
      if (i < 7) {
        read_x(i + 1);
        if (i == 3) scales(1);
        make_w(i + 1);
      }
#pragma unroll
      for (int f = 0; f < MT; ++f)
#pragma unroll
        for (int t = 0; t < NT; ++t)
          acc[f][t] =
              __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[i & 1][t], wf[i & 1][f], acc[f][t], 0, 0, 0);
      if (i < 7) {
#pragma unroll
        for (int k = 0; k < MT * NT; ++k) {
          if (k < NT) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);              // MFMA
          __builtin_amdgcn_sched_group_barrier(0x002, GT_VPM, 0);         // VALU
        }
      }
    }
  };
  auto arrive = [&](GtW<MT, F16> &w) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
#pragma unroll
    for (int f = 0; f < MT; ++f) {
      if constexpr (F16) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)"
                     : "+v"(w.q[f][0]), "+v"(w.q[f][1]), "+v"(w.q[f][2]), "+v"(w.q[f][3]),
                       "+v"(w.q[f][4]), "+v"(w.q[f][5]), "+v"(w.q[f][6]), "+v"(w.q[f][7])
                     ::"memory");
      } else {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)"
                     : "+v"(w.q[f][0]), "+v"(w.q[f][1]), "+v"(w.ix[f])::"memory");
      }
    }
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  GtW<MT, F16> w0, w1;
  load_x(step0, 0);
  load_w(step0, w0);
  const int last = step1 - 1;
  int st = step0;
  for (; st + 2 <= step1; st += 2) {
    arrive(w0);
    load_x(st + 1, 1);
    load_w(st + 1, w1);
    __builtin_amdgcn_sched_barrier(0);
    compute(w0, 0, st);
    arrive(w1);
    load_x(min(st + 2, last), 0);
    load_w(min(st + 2, last), w0);
    __builtin_amdgcn_sched_barrier(0);
    compute(w1, 1, st + 1);
  }
  if (st < step1) {
    arrive(w0);
    compute(w0, 0, st);
  }
  // the clamped look-ahead DMA lands in LDS nobody reads any more; it must
  // land before the block ends and its LDS is given away
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // acc[f][t][r]: token 32 t + 8 (r / 4) + 4 half + r % 4, weight row l32.
  // Stores go through a buffer over the output: an offset past its last token
  // (or the one given to lanes past the last row) is dropped by the range
  // check, so no store is under a branch.
  const uint32_t tok0 = (uint32_t)(t0 + wn * NT * 32 + 4 * half);
  if constexpr (EPI == GT_SWIGLU) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void *)y, 0, (int)((uint32_t)n * (uint32_t)out_f * 2u), 0x00020000);
    const int a = tm * (S::BM / 2) + (MT == 2 ? wm : wm % (S::WM / 2)) * 32 + l32;
    const uint32_t tb = (uint32_t)out_f * 2u;
    const uint32_t off0 = a < out_f ? tok0 * tb + (uint32_t)a * 2u : 0xC0000000u;
    auto store = [&](float g, float u, int t, int r) {
      __builtin_amdgcn_raw_buffer_store_b16(f2h(g / (1.0f + __expf(-g)) * u), rs,
                                            off0 + (uint32_t)(32 * t + 8 * (r >> 2) + (r & 3)) * tb,
                                            0, 0);
    };
    if constexpr (MT == 2) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) store(acc[0][t][r], acc[1][t][r], t, r);
    } else {
      // the up halves through LDS (16 bytes a lane, lanes adjacent)
      static_assert(S::WM / 2 * S::WN * NT * 4096 <= S::LDS, "the exchange reuses the x buffers");
      float *ex = (float *)gt_lds + (wn * (S::WM / 2) + wm % (S::WM / 2)) * (NT * 1024) + lane * 4;
      __syncthreads();
      if (wm >= S::WM / 2) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int r = 0; r < 16; r += 4)
            *(float4 *)(ex + t * 1024 + r * 64) = make_float4(acc[0][t][r], acc[0][t][r + 1],
                                                              acc[0][t][r + 2], acc[0][t][r + 3]);
      }
      __syncthreads();
      if (wm >= S::WM / 2) return;
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
          const float4 u = *(const float4 *)(ex + t * 1024 + r * 64);
          store(acc[0][t][r], u.x, t, r);
          store(acc[0][t][r + 1], u.y, t, r + 1);
          store(acc[0][t][r + 2], u.z, t, r + 2);
          store(acc[0][t][r + 3], u.w, t, r + 3);
        }
    }
    return;
  }
  if constexpr (EPI == GT_ROPE64 || EPI == GT_ROPE128) {
    // QK-norm, RoPE and the KV append of the wave's head, in the arithmetic of
    // gemm_reduce_rope_kernel (the two halves of a rotation pair are the
    // lane's two fragments); never split.
    static_assert(MT == 2, "a rotation pair");
    constexpr int HD = EPI == GT_ROPE64 ? 64 : 128, HALF = HD / 2;
    const int base = EPI == GT_ROPE64 ? tm * S::BM + wm * 64 : tm * S::BM + (wm >> 1) * 128;
    if (base >= out_f) return;  // a whole wave (out_f is whole heads); no barriers below
    const int h = base / HD, jj = EPI == GT_ROPE64 ? l32 : (wm & 1) * 32 + l32;
    const float b1 = bias ? h2f(bias[base + jj]) : 0.0f;
    const float b2 = bias ? h2f(bias[base + jj + HALF]) : 0.0f;
    const bool is_q = h < re.n_q, is_v = h >= re.n_q + re.n_kv;  // uniform in the wave
    const uint16_t *g = is_v ? nullptr : is_q ? re.q_norm_w : re.k_norm_w;
    const float g1 = g ? h2f(g[jj]) : 0.0f, g2 = g ? h2f(g[jj + HALF]) : 0.0f;
    const int kvh = is_v ? h - re.n_q - re.n_kv : h - re.n_q;
    // Rows of y and of the head's cache by buffer offsets: a token past n gets
    // an offset past the range and is dropped.
    const uint32_t tb = (uint32_t)out_f * 4u;
    const __amdgpu_buffer_rsrc_t yrs =
        __builtin_amdgcn_make_buffer_rsrc((void *)y, 0, (int)((uint32_t)n * tb), 0x00020000);
    const uint32_t yoff = tok0 * tb + (uint32_t)(base + jj) * 4u;
    const size_t head0 = (size_t)(is_q ? 0 : kvh) * re.max_seq + re.pos0;
    const __amdgpu_buffer_rsrc_t crs = __builtin_amdgcn_make_buffer_rsrc(
        (void *)((is_v ? re.v_cache : re.k_cache) + head0 * HD), 0,
        (int)((uint32_t)n * (uint32_t)(HD * 2)), 0x00020000);
    const uint32_t coff = tok0 * (uint32_t)(HD * 2) + (uint32_t)jj * 2u;
    const uint32_t rot = (uint32_t)(n * HALF * 4);  // the tokens' rows of the rotation tables
    const __amdgpu_buffer_rsrc_t cosr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(re.cos_tab + (size_t)re.pos0 * HALF), 0, (int)rot, 0x00020000);
    const __amdgpu_buffer_rsrc_t sinr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(re.sin_tab + (size_t)re.pos0 * HALF), 0, (int)rot, 0x00020000);
    const uint32_t roff = tok0 * (uint32_t)(HALF * 4) + (uint32_t)jj * 4u;
    auto store_f = [&](float v, uint32_t off) {
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), yrs, off, 0, 0);
    };
    if (is_v) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const uint32_t dt = (uint32_t)(32 * t + 8 * (r >> 2) + (r & 3));
          float x1 = acc[0][t][r], x2 = acc[1][t][r];
          if (bias) {
            x1 += b1;
            x2 += b2;
          }
          store_f(x1, yoff + dt * tb);
          store_f(x2, yoff + dt * tb + HALF * 4u);
          __builtin_amdgcn_raw_buffer_store_b16(f2h(x1), crs, coff + dt * (HD * 2u), 0, 0);
          __builtin_amdgcn_raw_buffer_store_b16(f2h(x2), crs, coff + dt * (HD * 2u) + HALF * 2u, 0, 0);
        }
      return;
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      uint32_t c[16], sn[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t dt = (uint32_t)(32 * t + 8 * (r >> 2) + (r & 3));
        c[r] = __builtin_amdgcn_raw_buffer_load_b32(cosr, roff + dt * (HALF * 4u), 0, 0);
        sn[r] = __builtin_amdgcn_raw_buffer_load_b32(sinr, roff + dt * (HALF * 4u), 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t dt = (uint32_t)(32 * t + 8 * (r >> 2) + (r & 3));
        float x1 = acc[0][t][r], x2 = acc[1][t][r];
        if (bias) {
          x1 += b1;
          x2 += b2;
        }
        const float k1 = x1, k2 = x2;  // a k row keeps the value as computed
        if (EPI == GT_ROPE64 && g) {
          const float ss = half_wave_sum(fmaf(x1, x1, x2 * x2));
          const float sc = 1.0f / sqrtf(ss / (float)HD + re.eps);
          x1 = x1 * sc * g1;
          x2 = x2 * sc * g2;
        }
        const float cv = __builtin_bit_cast(float, c[r]), sv = __builtin_bit_cast(float, sn[r]);
        const float lo = rope_lo(x1, x2, cv, sv), hi = rope_hi(x1, x2, cv, sv);
        store_f(is_q ? lo : k1, yoff + dt * tb);
        store_f(is_q ? hi : k2, yoff + dt * tb + HALF * 4u);
        if (!is_q) {
          __builtin_amdgcn_raw_buffer_store_b16(f2h(lo), crs, coff + dt * (HD * 2u), 0, 0);
          __builtin_amdgcn_raw_buffer_store_b16(f2h(hi), crs, coff + dt * (HD * 2u) + HALF * 2u, 0, 0);
        }
      }
    }
    return;
  }
  const bool split = ws != nullptr;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(split ? ws + (size_t)blockIdx.y * n * out_f : y), 0,
      (int)((uint32_t)n * (uint32_t)out_f * 4u), 0x00020000);
  const uint32_t tb = (uint32_t)out_f * 4u;
#pragma unroll
  for (int f = 0; f < MT; ++f) {
    const int r_ = tm * S::BM + (wm * MT + f) * 32 + l32;
    const uint32_t off0 = r_ < out_f ? tok0 * tb + (uint32_t)r_ * 4u : 0xC0000000u;
    const float bj = !split && bias ? h2f(bias[min(r_, out_f - 1)]) : 0.0f;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      uint32_t old[16];
      if (!split && accum) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          old[r] = __builtin_amdgcn_raw_buffer_load_b32(
              rs, off0 + (uint32_t)(32 * t + 8 * (r >> 2) + (r & 3)) * tb, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float v = acc[f][t][r];
        if (!split && bias) v += bj;
        if (!split && accum) v = __builtin_bit_cast(float, old[r]) + v;
        __builtin_amdgcn_raw_buffer_store_b32(
            __builtin_bit_cast(uint32_t, v), rs,
            off0 + (uint32_t)(32 * t + 8 * (r >> 2) + (r & 3)) * tb, 0, 0);
      }
    }
  }
}
