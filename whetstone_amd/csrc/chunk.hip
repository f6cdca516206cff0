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
// waves a SIMD (135 kept three: 77 against 65 us). Measured in us, calls in a row,
// against 16 or 32 tokens of one head a block with K and V staged through
// registers (heads, head_dim, tokens at position): 14/2 of 64, 4096 at 0: 71 ->
// 58; 14/2 of 64, 256 at 3840: 19.8 -> 16.9; 28/4 of 128, 243 at 1792: 29.0 ->
// 18.5; 28/4 of 128, 4096 at 0: 256 -> 215, 1000 at 0: 31.5 -> 26.9. Over few positions the
// launch's fixed parts count and the short kernel below is the faster one.
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
  // 2 G threads a row, four dims of every 8 G each. A row's weights, sum and
  // quotients are one chain for all of a thread's dims (two dims a thread in
  // 32 RW / 4 passes cost 0.4 us a pass: 28/4 heads of 128, 7 tokens at 0, 7.7
  // us whole; 6.6 now). 8-byte stores, or 2-byte ones where out starts
  // off 8 bytes.
  const bool whole_words = ((uintptr_t)out & 7u) == 0;
  const int live = min(32 * RW, rows - rb);
  constexpr int TPR = 2 * S::GROUPS, ND = HD / (4 * TPR);
  static_assert(S::THREADS == TPR * 32 * RW && ND * 4 * TPR == HD, "every dim once");
  const int r = tid / TPR, d0 = 4 * (tid % TPR);
  const float *p = mb + r * S::MR;
  float mw[S::GROUPS], M = -INFINITY, den = 0.0f;
  float4 num[ND];
#pragma unroll
  for (int k = 0; k < ND; ++k) num[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
  for (int w = 0; w < S::GROUPS; ++w) {
    mw[w] = p[w * 32 * RW * S::MR + HD];
    M = fmaxf(M, mw[w]);
  }
#pragma unroll
  for (int w = 0; w < S::GROUPS; ++w) {
    const float *pw = p + w * 32 * RW * S::MR;
    const float f = mw[w] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mw[w] - M);  // base 2
    den = fmaf(pw[HD + 1], f, den);
#pragma unroll
    for (int k = 0; k < ND; ++k) {
      const float4 v = *(const float4 *)(pw + d0 + 4 * TPR * k);
      num[k].x = fmaf(v.x, f, num[k].x);
      num[k].y = fmaf(v.y, f, num[k].y);
      num[k].z = fmaf(v.z, f, num[k].z);
      num[k].w = fmaf(v.w, f, num[k].w);
    }
  }
  if (r >= live) return;
  const int tk = (rb + r) / gqa, hd = kvh * gqa + (rb + r) % gqa;
  uint16_t *op = out + ((size_t)tk * n_q + hd) * HD + d0;
#pragma unroll
  for (int k = 0; k < ND; ++k, op += 4 * TPR) {
    const uint16_t h[4] = {f2h(num[k].x / den), f2h(num[k].y / den), f2h(num[k].z / den),
                           f2h(num[k].w / den)};
    if (whole_words)
      *(uint2 *)op = make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16),
                                (uint32_t)h[2] | ((uint32_t)h[3] << 16));
    else
#pragma unroll
      for (int i = 0; i < 4; ++i) op[i] = h[i];
  }
}

// ------------------------------------- chunk attention over few positions
//
// The same attention for a chunk over a short cache: a block per (query head,
// 16 tokens), four waves taking key tiles of 32 positions round-robin on
// v_mfma_f32_16x16x32_f16, K and V staged through registers, merged once
// through LDS. Its tile is a shorter chain than the kernel above (16 rows a wave
// instead of 32: half the MFMA time) on several times the blocks, which is what
// counts while a wave has a few tiles only. Scores, lazy maximum, P and the
// transposing V reads are those above; keys past the attended end read zeros
// through the buffer range check.
typedef float as_f4 __attribute__((ext_vector_type(4)));
typedef uint32_t as_u4 __attribute__((ext_vector_type(4)));

#define AS_WAVES 4

template <int HD>
struct AsShape {
  static constexpr int KS = HD / 32;              // k-steps of the scores
  static constexpr int NT = HD / 16;              // 16-dim output tiles
  static constexpr int VR = HD + 16;              // V row stride (halves)
  static constexpr int KR = HD + 8;               // K row stride (halves)
  static constexpr int VU = AC_KT * HD / 8 / 64;  // 16-byte K and V pieces per lane per tile
  static constexpr int TILES = AC_KT * VR + AC_KT * KR;
  static constexpr int MERGE = 16 * (HD + 2) * 2;  // the merge rows (floats), in halves
  static constexpr int WAVE = TILES > MERGE ? TILES : MERGE;
  static constexpr int LDS = AS_WAVES * WAVE * 2;
};

template <int HD, bool PLO>
__global__ __launch_bounds__(AS_WAVES * 64) void attn_chunk_short_kernel(
    const float *__restrict__ qkv, const uint16_t *__restrict__ k_cache,
    const uint16_t *__restrict__ v_cache, uint16_t *__restrict__ out, int n_q, int n_kv,
    int pos0, int n, int max_seq, float scale) {
  using S = AsShape<HD>;
  extern __shared__ __align__(16) unsigned char ac_lds[];
  // Token groups in reverse order: the longest blocks start first.
  const int head = blockIdx.x, t0 = (gridDim.y - 1 - blockIdx.y) * 16;
  const int kvh = head / (n_q / n_kv);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: the tile loop is scalar
  const int r16 = lane & 15, kg = lane >> 4;
  uint16_t *vs = (uint16_t *)ac_lds + wave * S::WAVE;  // V tile [AC_KT][VR], row-major
  uint16_t *ks = vs + AC_KT * S::VR;                   // K tile [AC_KT][KR], row-major
  const int stride_row = (n_q + 2 * n_kv) * HD;
  const uint16_t *kb = k_cache + (size_t)kvh * max_seq * HD;
  const uint16_t *vb = v_cache + (size_t)kvh * max_seq * HD;

  // q^T of token t0 + r16 as the B operand: dims 32s + 8kg + i, hi and lo
  const float qscale = scale * 1.44269504088896340736f;
  ac_h8 qh[S::KS], ql[S::KS];
  {
    const float *q = qkv + (size_t)min(t0 + r16, n - 1) * stride_row + (size_t)head * HD;
#pragma unroll
    for (int s = 0; s < S::KS; ++s) {
      const float4 a = *(const float4 *)(q + 32 * s + 8 * kg);
      const float4 b = *(const float4 *)(q + 32 * s + 8 * kg + 4);
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
  const int kend = min(pos0 + min(t0 + 16, n), max_seq);  // positions [0, kend) are attended
  const int ntiles = (kend + AC_KT - 1) / AC_KT;
  const int lim = pos0 + t0 + r16;  // the last position this lane's token attends

  // The whole byte offset goes in the vector offset, which is what the range
  // check compares with the buffer's size.
  const uint32_t kv_bytes = (uint32_t)kend * HD * 2u;
  const __amdgpu_buffer_rsrc_t krs =
      __builtin_amdgcn_make_buffer_rsrc((void *)kb, 0, (int)kv_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t vrs =
      __builtin_amdgcn_make_buffer_rsrc((void *)vb, 0, (int)kv_bytes, 0x00020000);
  const uint32_t voff = (uint32_t)lane * 16u;  // rows of a tile are contiguous
  as_u4 kr[S::VU], vr[S::VU];
  auto load_tile = [&](int kt) {
    const uint32_t so = (uint32_t)kt * (AC_KT * HD * 2);
#pragma unroll
    for (int j = 0; j < S::VU; ++j)
      kr[j] = __builtin_amdgcn_raw_buffer_load_b128(krs, so + voff + j * 1024, 0, 0);
#pragma unroll
    for (int j = 0; j < S::VU; ++j)
      vr[j] = __builtin_amdgcn_raw_buffer_load_b128(vrs, so + voff + j * 1024, 0, 0);
  };

  float m = -INFINITY, l = 0.0f;  // of the lane's token; l over this lane's keys
  as_f4 o[S::NT];                 // O^T: dims 16t + 4kg + i of token r16
#pragma unroll
  for (int t = 0; t < S::NT; ++t) o[t] = (as_f4){0.0f, 0.0f, 0.0f, 0.0f};

  load_tile(min(wave, ntiles - 1));
  for (int kt = wave; kt < ntiles; kt += AS_WAVES) {
    const int p0 = kt * AC_KT;
#pragma unroll
    for (int j = 0; j < S::VU; ++j) {
      const int u = lane + 64 * j, pr = u / (HD / 8), ch = u % (HD / 8);
      *(as_u4 *)(ks + pr * S::KR + 8 * ch) = kr[j];
      *(as_u4 *)(vs + pr * S::VR + 8 * ch) = vr[j];
    }
    // S^T for keys p0 + 16 t2 + 4kg + i of token r16
    as_f4 sc[2];
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      sc[t2] = (as_f4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < S::KS; ++s) {
        const ac_h8 a = *(const ac_h8 *)(ks + (16 * t2 + r16) * S::KR + 32 * s + 8 * kg);
        sc[t2] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, qh[s], sc[t2], 0, 0, 0);
        sc[t2] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, ql[s], sc[t2], 0, 0, 0);
      }
    }
    // the next tile's loads go out now (the registers above are consumed)
    load_tile(min(kt + AS_WAVES, ntiles - 1));
    // A tile wholly below the block's first token's limit needs no mask.
    if (!(p0 + AC_KT - 1 <= pos0 + t0 && p0 + AC_KT <= kend)) {  // uniform
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int p = p0 + 16 * t2 + 4 * kg + i;
          if (!(p <= lim && p < kend)) sc[t2][i] = -INFINITY;
        }
    }
#define AC_MAX(a, b) __builtin_elementwise_maximum(a, b)
    float mx = AC_MAX(AC_MAX(AC_MAX(sc[0][0], sc[0][1]), AC_MAX(sc[0][2], sc[0][3])),
                      AC_MAX(AC_MAX(sc[1][0], sc[1][1]), AC_MAX(sc[1][2], sc[1][3])));
    RowPair pr = xrow16(mx);  // the token's other keys: lanes r16 + 16 kg
    mx = AC_MAX(pr.a, pr.b);
    pr = xrow32(mx);
    mx = AC_MAX(pr.a, pr.b);
#undef AC_MAX
    // m moves only past m + 8; mx = -inf (no key of this token in the tile)
    // leaves it
    const bool bump = mx > m + 8.0f;
    const float mn = bump ? mx : m;
    const float corr = !bump ? 1.0f : m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mn);
    // finite, so that a token with no key yet (mn = -inf) gets 0, not NaN
    const float mref = mn == -INFINITY ? 0.0f : mn;
    ac_h8 ph, pl;
    float psum = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float p = __builtin_amdgcn_exp2f(sc[j >> 2][j & 3] - mref);
      psum += p;
      const _Float16 h = (_Float16)p;
      ph[j] = h;
      if constexpr (PLO) pl[j] = (_Float16)(p - (float)h);
    }
    l = l * corr + psum;
    m = mn;
    if (!__all(corr == 1.0f)) {
#pragma clang loop unroll(full)
      for (int t = 0; t < S::NT; ++t)
#pragma clang loop unroll(full)
        for (int i = 0; i < 4; ++i) o[t][i] *= corr;
    }
    // V^T operand: lane s of a 16-lane group reads key rows 4kg + s/4 and
    // 16 + 4kg + s/4, dims 16t + 4(s%4)
    const uint16_t *va = vs + (4 * kg + (r16 >> 2)) * S::VR + 4 * (r16 & 3);
#pragma clang loop unroll(full)
    for (int t = 0; t < S::NT; ++t) {
      const ac_h8 v = tr_pair((const unsigned char *)(va + 16 * t),
                              (const unsigned char *)(va + 16 * S::VR + 16 * t));
      o[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, ph, o[t], 0, 0, 0);
      if constexpr (PLO) o[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, pl, o[t], 0, 0, 0);
    }
  }

  // merge the waves: per wave (m, l, O[HD]) of its 16 tokens, in its own region
  float *mb = (float *)vs;
  {
    RowPair pr = xrow16(l);
    const float l2 = pr.a + pr.b;
    pr = xrow32(l2);
    if (kg == 0) {
      mb[r16 * (HD + 2)] = m;
      mb[r16 * (HD + 2) + 1] = pr.a + pr.b;
    }
#pragma unroll
    for (int t = 0; t < S::NT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) mb[r16 * (HD + 2) + 2 + 16 * t + 4 * kg + i] = o[t][i];
  }
  __syncthreads();
  const int rows = min(16, n - t0);
  for (int idx = tid; idx < rows * HD; idx += AS_WAVES * 64) {
    const int row = idx / HD, d = idx % HD;
    const float *p = (const float *)ac_lds + row * (HD + 2);
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < AS_WAVES; ++w) M = fmaxf(M, p[w * (S::WAVE / 2)]);
    float num = 0.0f, den = 0.0f;
#pragma unroll
    for (int w = 0; w < AS_WAVES; ++w) {
      const float *wb = p + w * (S::WAVE / 2);
      const float f = wb[0] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(wb[0] - M);  // base 2
      num = fmaf(wb[2 + d], f, num);
      den = fmaf(wb[1], f, den);
    }
    out[(size_t)(t0 + row) * n_q * HD + (size_t)head * HD + d] = f2h(num / den);
  }
}

template <int HD, bool PLO>
static void attn_chunk_short(const void *qkv, const void *k_cache, const void *v_cache, void *out,
                             int n_q, int n_kv, int pos0, int n, int max_seq, float scale) {
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute((const void *)attn_chunk_short_kernel<HD, PLO>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, AsShape<HD>::LDS);
    attr = true;
  }
  attn_chunk_short_kernel<HD, PLO>
      <<<dim3(n_q, (n + 15) / 16), AS_WAVES * 64, AsShape<HD>::LDS, WST_STREAM>>>(
          (const float *)qkv, (const uint16_t *)k_cache, (const uint16_t *)v_cache,
          (uint16_t *)out, n_q, n_kv, pos0, n, max_seq, scale);
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
  // A call by itself (plan_n 0: no other launch has to give its tokens the same
  // bits) over few positions: us, short kernel / this one, 28/4 heads of 128:
  // 7 tokens at 100 5.5 / 6.8, at 645 8.5 / 10.1, at 1000 11.9 / 11.5; 128 at 100
  // 7.0 / 7.8, at 300 9.1 / 9.0; 256 at 0 8.3 / 7.7. 14/2 of 64: 16 at 300 5.4 /
  // 6.7, at 1500 9.4 / 9.7, at 2200 12.2 / 11.6; 256 at 1000 8.9 / 9.3, at 1500
  // 10.6 / 10.5.
  if (plan_n <= 0) {
    if (n < 512 && (HD == 64 ? pos0 + 2 * n < 1700 : pos0 + 4 * n < 680)) {
      (plo ? attn_chunk_short<HD, true> : attn_chunk_short<HD, false>)(
          qkv, k_cache, v_cache, out, n_q, n_kv, pos0, n, max_seq, scale);
      return;
    }
    plan_n = n;
  }
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
  const int pn = plan_n <= 0 ? 0 : plan_n < n ? plan_n : n;
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
                         0);
}
