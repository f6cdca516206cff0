// Multi-token ("chunk") forms of the decode step, for prefill.
// reference: crates/whetstone-kernels/cuda/chunk_gemm.cu, chunk_ops.cu.
//
// Activations are token-major [n][dim]; pos0 is passed by value (a chunk pass
// is not graph-captured, chunk.rs:1-12). Causality is the loop bound: token j
// attends to cache positions [0, pos0 + j].
#include "common.hpp"

#define CHUNK_MAX_TOKENS 256

extern "C" int32_t wst_chunk_max_tokens(void) { return CHUNK_MAX_TOKENS; }

// Implemented in gemm.hip (MFMA).
wst_status_t wst_gemm_mfma(bool hier, const void *w, const void *si, const void *sb,
                           const void *x, const void *bias, void *y, int32_t in_f, int32_t out_f,
                           int32_t n, int32_t accum, float *ws_ext = nullptr, size_t ws_cap = 0,
                           int32_t plan_n = 0);

extern "C" wst_status_t wst_gemm_int4_hier_chunks(const void *qw, const void *si, const void *sb,
                                                  const void *x, const void *bias, void *y,
                                                  int32_t in_f, int32_t out_f, int32_t n,
                                                  int32_t accum, int32_t plan_n) {
  WST_REQUIRE(qw && si && sb && x && y, "wst_gemm_int4_hier: null pointer");
  WST_REQUIRE(in_f > 0 && out_f > 0 && n > 0, "wst_gemm_int4_hier: non-positive dimension");
  WST_REQUIRE(in_f % 32 == 0, "wst_gemm_int4_hier: in_features must be a multiple of 32");
  WST_REQUIRE(!(((uintptr_t)qw | (uintptr_t)x) & 15u),
              "wst_gemm_int4_hier: qw and x must be 16-byte aligned");
  const wst_status_t st =
      wst_gemm_mfma(true, qw, si, sb, x, bias, y, in_f, out_f, n, accum, nullptr, 0, plan_n);
  if (st != WST_OK) return st;
  WST_TRY_KERNEL("wst_gemm_int4_hier");
  return WST_OK;
}

extern "C" wst_status_t wst_gemm_int4_hier(const void *qw, const void *si, const void *sb,
                                           const void *x, const void *bias, void *y,
                                           int32_t in_f, int32_t out_f, int32_t n,
                                           int32_t accum) {
  return wst_gemm_int4_hier_chunks(qw, si, sb, x, bias, y, in_f, out_f, n, accum, n);
}

extern "C" wst_status_t wst_gemm_fp16(const void *w, const void *x, const void *bias, void *y,
                                      int32_t in_f, int32_t out_f, int32_t n, int32_t accum) {
  WST_REQUIRE(w && x && y, "wst_gemm_fp16: null pointer");
  WST_REQUIRE(in_f > 0 && out_f > 0 && n > 0, "wst_gemm_fp16: non-positive dimension");
  WST_REQUIRE(in_f % 8 == 0, "wst_gemm_fp16: in_features must be a multiple of 8");
  if (in_f % 32 == 0 && !(((uintptr_t)w | (uintptr_t)x) & 15u)) {
    const wst_status_t st = wst_gemm_mfma(false, w, nullptr, nullptr, x, bias, y, in_f, out_f, n,
                                          accum);
    if (st != WST_OK) return st;
    WST_TRY_KERNEL("wst_gemm_fp16");
    return WST_OK;
  }
  for (int j = 0; j < n; ++j) {  // widths that are not whole 32-column steps
    const wst_status_t st = wst_gemv_fp16_ex(w, (const uint16_t *)x + (size_t)j * in_f, bias,
                                             (float *)y + (size_t)j * out_f, in_f, out_f, accum);
    if (st != WST_OK) return st;
  }
  return WST_OK;
}

// Causal chunk attention (chunk_ops.cu:187-265) for head_dim 256: one block
// per (query head, token). q is the rotated q of the token's qkv row; the cache already holds
// the chunk's own k/v (wst_rope_cache_chunk ran first). Each of the 4 waves
// sweeps every 4th position with head_dim/64 elements per lane and its own
// online softmax; the waves merge through LDS.
template <int HD>
__global__ __launch_bounds__(256) void attn_chunk_kernel(
    const float *__restrict__ qkv, const uint16_t *__restrict__ k_cache,
    const uint16_t *__restrict__ v_cache, uint16_t *__restrict__ out, int n_q, int n_kv,
    int pos0, int max_seq, float scale) {
  constexpr int EPL = HD / 64;  // elements per lane
  const int head = blockIdx.x, tok = blockIdx.y;
  const int gqa = n_q / n_kv, kvh = head / gqa;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int stride_row = (n_q + 2 * n_kv) * HD;
  const float *q = qkv + (size_t)tok * stride_row + (size_t)head * HD;
  const int seq = min(pos0 + tok + 1, max_seq);

  float qr[EPL], acc[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    qr[e] = q[lane + 64 * e] * scale;
    acc[e] = 0.0f;
  }
  float m = -INFINITY, l = 0.0f;
  const uint16_t *kb = k_cache + (size_t)kvh * max_seq * HD;
  const uint16_t *vb = v_cache + (size_t)kvh * max_seq * HD;
  for (int t = wave; t < seq; t += 4) {
    float s = 0.0f;
#pragma unroll
    for (int e = 0; e < EPL; ++e) s = fmaf(qr[e], h2f(kb[(size_t)t * HD + lane + 64 * e]), s);
    s = wave_sum(s);
    const float mn = fmaxf(m, s);
    const float corr = __expf(m - mn);
    const float p = __expf(s - mn);
    l = fmaf(l, corr, p);
#pragma unroll
    for (int e = 0; e < EPL; ++e)
      acc[e] = fmaf(p, h2f(vb[(size_t)t * HD + lane + 64 * e]), acc[e] * corr);
    m = mn;
  }
  __shared__ float sm[4][HD + 2];
#pragma unroll
  for (int e = 0; e < EPL; ++e) sm[wave][2 + lane + 64 * e] = acc[e];
  if (lane == 0) {
    sm[wave][0] = m;
    sm[wave][1] = l;
  }
  __syncthreads();
  for (int d = tid; d < HD; d += 256) {
    float M = -INFINITY;
    for (int w = 0; w < 4; ++w) M = fmaxf(M, sm[w][0]);
    float num = 0.0f, den = 0.0f;
    for (int w = 0; w < 4; ++w) {
      const float f = (sm[w][0] == -INFINITY) ? 0.0f : __expf(sm[w][0] - M);
      num = fmaf(sm[w][2 + d], f, num);
      den = fmaf(sm[w][1], f, den);
    }
    out[(size_t)tok * n_q * HD + (size_t)head * HD + d] = f2h(num / den);
  }
}

// ------------------------------------------------------ MFMA chunk attention
//
// The same causal attention (chunk_ops.cu:187-265) as flash attention on
// v_mfma_f32_32x32x16_f16, for head_dim 64 and 128, in transposed form:
// S^T = K . q^T and O^T = V^T . P^T, keys on the MFMA's M side and query rows
// on its N side.
// * A query row is a (token, head) pair of one kv head, token-major, so the
//   heads that share a kv head share its K and V tiles. A wave holds 32 rows;
//   a block holds RW row waves times G key groups. Group g takes the key tiles
//   of 32 positions g, g + G, .. with its own online softmax, its RW waves
//   sharing the tile in LDS, and the groups merge once at the end.
// * K and V tiles go memory -> LDS by DMA (global_load_lds_dwordx4), one tile
//   ahead in two buffers: no registers, no LDS writes by the waves. Rows past
//   the block's last attended position re-read that position (their scores are
//   masked), so nothing past it is read. A row's 16-byte chunk c sits at slot
//   c ^ f(key), with f such that the 16 lanes of an operand read touch all 64
//   banks once.
// * A lane holds one query row and 16 of the tile's keys. Scores: q (already
//   rotated, times log2(e)/sqrt(hd), so the softmax is in base 2) enters as its
//   f16 hi part plus the f16 rounding of the rest, so the products keep ~22
//   bits.
// * The row's reference maximum m enters as the score MFMA's C operand (-m),
//   so the accumulators are s - m as they come. m moves only when a tile's
//   maximum passes it by more than 8 (base 2): the exponentials stay at most
//   2^8, far inside f16 and f32, and the tile's common path is 8 three-way
//   maxima, one wave-uniform test, 16 exponentials, 16 adds and 8 packed
//   conversions: about 60 VALU ops a tile where the form with a maximum,
//   subtraction and rescale test per row took 180. Softmax is exact for any
//   reference point; only roundings move.
// * P^T never goes through LDS: the exponentials, rounded to f16, are the B
//   operand of O^T = V^T . P^T as they stand, the MFMA's K index k = 8 h + j
//   (h = lane / 32) standing for key 4 h + j (j < 4) and 8 + 4 h + j - 4
//   (j >= 4) of 16; the V^T operand is gathered in that key order by the
//   gfx950 transposing LDS read (ds_read_b64_tr_b16: within 16 lanes, lane L's
//   element i comes from lane 4i + L/4's element L%4).
// * P in one f16 (round to nearest, relative error <= 2^-11 per weight,
//   averaging over the keys) where q keeps its hi + lo parts: a score error
//   is an exponent error, a P error only a weight error, and the output is
//   rounded to f16 (2^-11) anyway. WST_ATTN_CHUNK_PLO=1 adds P's low part.
// Causality is a mask: token j keeps positions <= pos0 + j.
//
// A row's result does not depend on RW: its valid keys fall in the same
// tiles, taken by the same group in the same order (a block's extra tiles are
// wholly masked for it: no term and no rescale), so RW is picked by the row
// count alone (WST_ATTN_CHUNK_TG=1|2 forces one).
//
// What bounds it: a tile's dependent chain (LDS reads, the score MFMAs into one
// accumulator, exponentials, P.V: about 0.5 us for a wave alone) where a CU
// holds few waves, and MFMA and VALU issue (12 32-clk MFMAs and ~100 VALU ops a
// tile at head_dim 64) where it is full: 128 VGPRs at head_dim 64 keep four
// waves a SIMD (135 kept three: 77 against 65 us). Measured in us against 16 or
// 32 tokens of one head a block with K and V staged through registers (heads,
// head_dim, tokens at position): 14/2 of 64, 4096 at 0: 79 -> 63; 14/2 of 64,
// 256 at 3840: 21.8 -> 18.3; 28/4 of 128, 243 at 1792: 33 -> 21; 28/4 of 128,
// 4096 at 0: 285 -> 245, 1000 at 0: 39 -> 33. A short prompt's one or two
// tiles pay 0.8 us more for the merge (100 tokens at 0: 4.7 -> 5.5).
typedef _Float16 ac_h8 __attribute__((ext_vector_type(8)));
typedef short ac_s4 __attribute__((ext_vector_type(4)));
typedef float ac_f16v __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) ac_s4 ac_lds_s4;

#define AC_KT 32  // key positions per tile

template <int HD, int RW, int GROUPS_>
struct AcShape {
  static constexpr int GROUPS = GROUPS_;         // key groups
  static constexpr int KS = HD / 16;             // k-steps of the scores
  static constexpr int NF = HD / 32;             // 32-dim output fragments
  static constexpr int ROW = HD * 2;             // bytes of a K or V row
  static constexpr int TILE = AC_KT * ROW;       // bytes of a K (or V) tile
  static constexpr int DMA = TILE / 1024 / RW;   // 1 KB ops a wave issues per tile, K and V each
  static constexpr int THREADS = 64 * GROUPS * RW;
  static constexpr int LDS_T = GROUPS * 2 * 2 * TILE;
  static constexpr int MR = HD + 4;              // floats of a merge row: O, m, l
  static constexpr int LDS_M = GROUPS * RW * 32 * MR * 4;
  static constexpr int LDS = LDS_T > LDS_M ? LDS_T : LDS_M;
  static_assert(LDS <= 160 * 1024, "one CU's LDS");
};

// Slot of chunk c in key row `key` of a K or V tile (rows of 8 or 16 chunks).
template <int HD>
__device__ __forceinline__ int ac_kswz(int key) {
  return HD == 64 ? (key >> 1) & 7 : key & 15;  // 16 keys, one chunk: 16 slots of 64 banks
}
template <int HD>
__device__ __forceinline__ int ac_vswz(int key) {
  return HD == 64 ? (key & 2) << 1 : (key & 3) << 2;  // 4 keys, 4 chunks: 16 slots
}

// Eight halves as an MFMA operand from two transposing reads.
__device__ __forceinline__ ac_h8 tr_pair(const unsigned char *a0, const unsigned char *a1) {
  const ac_s4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ac_lds_s4 *)a0);
  const ac_s4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ac_lds_s4 *)a1);
  return __builtin_bit_cast(ac_h8, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int HD, int RW, int G, bool PLO>
__global__ __launch_bounds__((64 * RW * G), (HD == 64 ? 4 : 2)) void attn_chunk_mfma_kernel(
    const float *__restrict__ qkv, const uint16_t *__restrict__ k_cache,
    const uint16_t *__restrict__ v_cache, uint16_t *__restrict__ out, int n_q, int n_kv,
    int pos0, int n, int max_seq, float scale) {
  using S = AcShape<HD, RW, G>;
  extern __shared__ __align__(16) unsigned char ac_lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: the tile loop is scalar
  const int grp = wave / RW, rw = wave % RW;
  const int l32 = lane & 31, half = lane >> 5;
  const int gqa = n_q / n_kv, rows = n * gqa;
  // Row blocks in reverse order: blocks are dispatched in index order, and the
  // last rows attend to the most positions, so the longest blocks start first
  // and the short ones fill in behind them.
  const int kvh = blockIdx.x % n_kv;
  const int rb = (gridDim.x / n_kv - 1 - blockIdx.x / n_kv) * (32 * RW);  // the block's first row
  const int r0 = rb + 32 * rw;                                           // the wave's
  const int stride_row = (n_q + 2 * n_kv) * HD;
  const int row = min(r0 + l32, rows - 1), tok = row / gqa;

  // Positions [0, kend) are attended by some row of the block, [0, wend) by
  // some row of the wave, and [0, wall) by every one of them.
  const int kend = min(pos0 + (min(rb + 32 * RW, rows) - 1) / gqa + 1, max_seq);
  const int wend = r0 < rows ? min(pos0 + (min(r0 + 32, rows) - 1) / gqa + 1, max_seq) : 0;
  const int wall = min(pos0 + min(r0, rows - 1) / gqa + 1, max_seq);
  const int lim = pos0 + tok;  // the last position this lane's row attends
  const int iters = ((kend + AC_KT - 1) / AC_KT + S::GROUPS - 1) / S::GROUPS;

  // DMA of tile kt into buffer buf: op i of this wave covers 1024 / ROW key
  // rows from (rw * DMA + i) * 1024 / ROW on.
  const char *kb = (const char *)(k_cache + (size_t)kvh * max_seq * HD);
  const char *vb = (const char *)(v_cache + (size_t)kvh * max_seq * HD);
  const uint32_t lds0 = (uint32_t)(uintptr_t)ac_lds + (uint32_t)grp * (4 * S::TILE);
  constexpr int RPO = 1024 / S::ROW, CPR = S::ROW / 16;  // rows per op, chunks per row
  const int dr = lane / CPR, dp = lane % CPR;
  auto load_tile = [&](int kt, int buf) {
    const uint32_t dst = lds0 + (uint32_t)buf * (2 * S::TILE) + (uint32_t)rw * (S::DMA * 1024u);
#pragma unroll
    for (int i = 0; i < S::DMA; ++i) {
      const int key = (rw * S::DMA + i) * RPO + dr;
      const uint32_t at = (uint32_t)min(kt * AC_KT + key, kend - 1) * (uint32_t)S::ROW;
      const uint32_t ko = at + (uint32_t)((dp ^ ac_kswz<HD>(key)) * 16);
      const uint32_t vo = at + (uint32_t)((dp ^ ac_vswz<HD>(key)) * 16);
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                   ::"s"(dst + i * 1024u), "v"(ko), "s"(kb) : "memory");
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                   ::"s"(dst + S::TILE + i * 1024u), "v"(vo), "s"(vb) : "memory");
    }
  };

  load_tile(grp, 0);

  // q^T of the lane's row as the B operand: dims 16s + 8 half + i, hi and lo
  const float qscale = scale * 1.44269504088896340736f;
  ac_h8 qh[S::KS], ql[S::KS];
  {
    const float *q = qkv + (size_t)tok * stride_row + (size_t)(kvh * gqa + row % gqa) * HD;
#pragma unroll
    for (int s = 0; s < S::KS; ++s) {
      const float4 a = *(const float4 *)(q + 16 * s + 8 * half);
      const float4 b = *(const float4 *)(q + 16 * s + 8 * half + 4);
      const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float x = v[i] * qscale;
        const _Float16 h = (_Float16)x;
        qh[s][i] = h;
        ql[s][i] = (_Float16)(x - (float)h);
      }
    }
  }
  float l = 0.0f, m = -INFINITY;  // of the lane's row; l over this lane's keys
  float thr = -INFINITY;          // a tile maximum (of s - m) above it moves m
  ac_f16v negm;                   // -m in every register (0 while there is no m)
  ac_f16v o[S::NF];               // O^T: dims 32f + 8(i/4) + 4 half + i%4 of row l32
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    negm[i] = 0.0f;
#pragma unroll
    for (int f = 0; f < S::NF; ++f) o[f][i] = 0.0f;
  }
  const uint32_t gbase = (uint32_t)grp * (4 * S::TILE);
  const uint32_t krow = gbase + (uint32_t)(l32 * S::ROW);
  const int ksw = ac_kswz<HD>(l32) ^ half;  // chunk 2s + half of key l32: slot ksw ^ 2s
  // V^T operand rows: key 4 half + (l16 / 4), dims 16 (lane / 16 % 2) + 4 (l16 % 4)
  const int l16 = lane & 15, vkey = 4 * half + (l16 >> 2);
  const int vch = 2 * ((lane >> 4) & 1) + ((l16 & 3) >> 1);
  const uint32_t vrow = gbase + S::TILE + (uint32_t)(vkey * S::ROW + 8 * (l16 & 1));

  for (int it = 0; it < iters; ++it) {
    // The tile has landed (this wave's part; with the barrier every part), and
    // the group is done with the other buffer.
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    if constexpr (RW > 1) __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const int kt = it * S::GROUPS + grp, p0 = kt * AC_KT;
    if (it + 1 < iters) load_tile(kt + S::GROUPS, (it + 1) & 1);
    if (p0 >= wend) continue;  // every row of the wave masked: no term
    const uint32_t bo = (uint32_t)((it & 1) * 2) * S::TILE;
    // S^T - m: keys p0 + 8(i/4) + 4 half + i%4 of row l32
    ac_f16v sc = negm;
#pragma unroll
    for (int s = 0; s < S::KS; ++s) {
      const ac_h8 a = *(const ac_h8 *)(ac_lds + bo + krow + (uint32_t)((ksw ^ (2 * s)) * 16));
      sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qh[s], sc, 0, 0, 0);
      sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, ql[s], sc, 0, 0, 0);
    }
    if (p0 + AC_KT > wall) {  // uniform: some row's limit is inside the tile
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int p = p0 + 8 * (i >> 2) + 4 * half + (i & 3);
        if (!(p <= lim && p < kend)) sc[i] = -INFINITY;
      }
    }
#define AC_MAX(a, b) __builtin_elementwise_maximum(a, b)
    float mx = sc[0];
#pragma unroll
    for (int i = 1; i < 15; i += 2) mx = AC_MAX(AC_MAX(mx, sc[i]), sc[i + 1]);
    mx = AC_MAX(mx, sc[15]);
    // (a NaN score compares false: it stays in sc and reaches the output)
    if (__any(mx > thr)) {
      const RowPair pr = xrow32(mx);  // the row's other keys
      mx = AC_MAX(pr.a, pr.b);
      const bool bump = mx > thr;
      const float d = bump ? mx : 0.0f;
      const float corr = !bump ? 1.0f : m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(-d);
      m = !bump ? m : m == -INFINITY ? d : m + d;
      thr = bump ? 8.0f : thr;
      l *= corr;
      const float nm = m == -INFINITY ? 0.0f : -m;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        sc[i] -= d;
        negm[i] = nm;
#pragma unroll
        for (int f = 0; f < S::NF; ++f) o[f][i] *= corr;
      }
    }
#undef AC_MAX
    ac_h8 ph[2], pl[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float p = __builtin_amdgcn_exp2f(sc[i]);  // 0 for a masked score
      l += p;
      const _Float16 h = (_Float16)p;
      ph[i >> 3][i & 7] = h;
      if constexpr (PLO) pl[i >> 3][i & 7] = (_Float16)(p - (float)h);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int f = 0; f < S::NF; ++f) {
        // keys 16u + vkey and 16u + 8 + vkey, chunk 4f + vch: the swizzle of
        // both keys is vkey's (it has period 4)
        const unsigned char *va = ac_lds + bo + vrow + (uint32_t)(16 * u * S::ROW) +
                                  (uint32_t)(((4 * f + vch) ^ ac_vswz<HD>(vkey)) * 16);
        const ac_h8 v = tr_pair(va, va + 8 * S::ROW);
        o[f] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v, ph[u], o[f], 0, 0, 0);
        if constexpr (PLO) o[f] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v, pl[u], o[f], 0, 0, 0);
      }
  }

  // merge the groups: per row (m, l, O[HD])
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __syncthreads();
  float *mb = (float *)ac_lds;  // [S::GROUPS][32 RW][MR]
  {
    const RowPair pr = xrow32(l);
    float *w = mb + (grp * 32 * RW + 32 * rw + l32) * S::MR;
    if (half == 0) {
      w[HD] = m;
      w[HD + 1] = pr.a + pr.b;
    }
#pragma unroll
    for (int f = 0; f < S::NF; ++f)
#pragma unroll
      for (int i = 0; i < 16; i += 4)
        *(float4 *)(w + 32 * f + 2 * i + 4 * half) =
            make_float4(o[f][i], o[f][i + 1], o[f][i + 2], o[f][i + 3]);
  }
  __syncthreads();
  // Two dims a thread, 4-byte stores.
  const int live = min(32 * RW, rows - rb);
  constexpr int PER = S::THREADS / (HD / 2);  // rows a pass
  const int d = 2 * (tid % (HD / 2));
#pragma unroll
  for (int k = 0; k < 32 * RW / PER; ++k) {
    const int r = tid / (HD / 2) + k * PER;
    if (r >= live) continue;
    const float *p = mb + r * S::MR;
    float mw[S::GROUPS], M = -INFINITY;
#pragma unroll
    for (int w = 0; w < S::GROUPS; ++w) {
      mw[w] = p[w * 32 * RW * S::MR + HD];
      M = fmaxf(M, mw[w]);
    }
    float n0 = 0.0f, n1 = 0.0f, den = 0.0f;
#pragma unroll
    for (int w = 0; w < S::GROUPS; ++w) {
      const float *pw = p + w * 32 * RW * S::MR;
      const float2 v = *(const float2 *)(pw + d);
      const float f = mw[w] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mw[w] - M);  // base 2
      n0 = fmaf(v.x, f, n0);
      n1 = fmaf(v.y, f, n1);
      den = fmaf(pw[HD + 1], f, den);
    }
    const int tk = (rb + r) / gqa, hd = kvh * gqa + (rb + r) % gqa;
    *(uint32_t *)(out + ((size_t)tk * n_q + hd) * HD + d) =
        (uint32_t)f2h(n0 / den) | ((uint32_t)f2h(n1 / den) << 16);
  }
}

template <int HD, int RW, int G, bool PLO>
static void attn_chunk_mfma_rw(const void *qkv, const void *k_cache, const void *v_cache, void *out,
                               int n_q, int n_kv, int pos0, int n, int max_seq, float scale) {
  using S = AcShape<HD, RW, G>;
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute((const void *)attn_chunk_mfma_kernel<HD, RW, G, PLO>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS);
    attr = true;
  }
  const int rows = n * (n_q / n_kv);
  attn_chunk_mfma_kernel<HD, RW, G, PLO>
      <<<n_kv * ((rows + 32 * RW - 1) / (32 * RW)), S::THREADS, S::LDS, WST_STREAM>>>(
          (const float *)qkv, (const uint16_t *)k_cache, (const uint16_t *)v_cache,
          (uint16_t *)out, n_q, n_kv, pos0, n, max_seq, scale);
}

// Two row waves a group (64 query rows a block) where that still gives every
// CU a block; one (32 rows) below. Eight key groups instead of four for a
// chunk's worth of tokens at head_dim 64 (at 128 their tiles would not fit one
// CU's LDS): few blocks, so the length of a wave's tile chain is what counts
// (14/2 heads of 64, 256 tokens at 3840: 22.5 -> 18.2 us; 4096 tokens from 0:
// 65 us with four, 82 with eight). The group count decides a row's sum order,
// so it goes by plan_n, the token count the caller plans for (up to four tiles
// the fifth group and on are empty and change nothing).
template <int HD>
static void attn_chunk_mfma(const void *qkv, const void *k_cache, const void *v_cache, void *out,
                            int n_q, int n_kv, int pos0, int n, int max_seq, float scale,
                            int plan_n) {
  const char *v = getenv("WST_ATTN_CHUNK_TG"), *pv = getenv("WST_ATTN_CHUNK_PLO");
  const bool plo = pv && pv[0] == '1';  // P as f16 hi + lo
  const int rows = n * (n_q / n_kv);
  const bool two = v && (v[0] == '1' || v[0] == '2') ? v[0] == '2'
                                                     : n_kv * ((rows + 63) / 64) >= wst_cu_count();
  auto go = two ? (plo ? attn_chunk_mfma_rw<HD, 2, 4, true> : attn_chunk_mfma_rw<HD, 2, 4, false>)
                : (plo ? attn_chunk_mfma_rw<HD, 1, 4, true> : attn_chunk_mfma_rw<HD, 1, 4, false>);
  if constexpr (HD == 64)
    if (plan_n <= CHUNK_MAX_TOKENS && pos0 + n > 4 * AC_KT)
      go = two ? (plo ? attn_chunk_mfma_rw<HD, 2, 8, true> : attn_chunk_mfma_rw<HD, 2, 8, false>)
               : (plo ? attn_chunk_mfma_rw<HD, 1, 8, true> : attn_chunk_mfma_rw<HD, 1, 8, false>);
  go(qkv, k_cache, v_cache, out, n_q, n_kv, pos0, n, max_seq, scale);
}

extern "C" wst_status_t wst_attn_chunks(const void *qkv, const void *k_cache, const void *v_cache,
                                        void *out, int32_t n_q, int32_t n_kv, int32_t head_dim,
                                        int32_t pos0, int32_t n, int32_t max_seq, float scale,
                                        int32_t plan_n) {
  const int pn = plan_n > 0 && plan_n < n ? plan_n : n;
  WST_REQUIRE(qkv && k_cache && v_cache && out, "wst_attn_chunk: null pointer");
  WST_REQUIRE(n_q > 0 && n_kv > 0 && n_q % n_kv == 0 && n > 0 && n <= 65535,
              "wst_attn_chunk: bad shape");
  WST_REQUIRE(max_seq > 0 && pos0 >= 0 && pos0 + n <= max_seq,
              "wst_attn_chunk: chunk does not fit the cache");
  WST_REQUIRE(!(((uintptr_t)qkv | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15u),
              "wst_attn_chunk: qkv and the caches must be 16-byte aligned");
  // The MFMA kernel addresses a head's cache rows with 32-bit buffer offsets.
  WST_REQUIRE((int64_t)max_seq * head_dim * 2 < ((int64_t)1 << 31),
              "wst_attn_chunk: a head's cache rows exceed 2 GiB");
  const dim3 grid(n_q, n);
  switch (head_dim) {
    case 64:
      attn_chunk_mfma<64>(qkv, k_cache, v_cache, out, n_q, n_kv, pos0, n, max_seq, scale, pn);
      break;
    case 128:
      attn_chunk_mfma<128>(qkv, k_cache, v_cache, out, n_q, n_kv, pos0, n, max_seq, scale, pn);
      break;
    case 256:
      attn_chunk_kernel<256><<<grid, 256, 0, WST_STREAM>>>(
          (const float *)qkv, (const uint16_t *)k_cache, (const uint16_t *)v_cache,
          (uint16_t *)out, n_q, n_kv, pos0, max_seq, scale);
      break;
    default:
      WST_REQUIRE(false, "wst_attn_chunk: head_dim must be 64, 128 or 256");
  }
  WST_TRY_KERNEL("wst_attn_chunk");
  return WST_OK;
}

extern "C" wst_status_t wst_attn_chunk(const void *qkv, const void *k_cache, const void *v_cache,
                                       void *out, int32_t n_q, int32_t n_kv, int32_t head_dim,
                                       int32_t pos0, int32_t n, int32_t max_seq, float scale) {
  return wst_attn_chunks(qkv, k_cache, v_cache, out, n_q, n_kv, head_dim, pos0, n, max_seq, scale,
                         n);
}
