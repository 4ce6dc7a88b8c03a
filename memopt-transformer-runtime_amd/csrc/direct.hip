// direct.hip — multi-query paged attention for short query blocks, straight
// from the cache to the matrix cores (gfx950): no staging launch, no staged
// copy of K and V, no LDS for operands.
//
// Semantics: those of prefill.hip (TheRadDani/memopt-transformer-runtime
// src/csrc/attention.cu:98-339 with sinks, and the causal rule of
// scripts/bench_accuracy.py:253-280), over INT4 page pools, the reference's
// token-major INT4 codes with separate scales, and fp16 pools. INT4 elements
// become fp16(RN((code - 8) * scale)), the values of the reference's
// dequantize kernel (src/csrc/quantization.cu:232-270).
//
// Why a second multi-query path: with a few queries per sequence the call is
// bound by the cache bytes, like a decode, but the staged path writes and
// re-reads 8 bytes of fp16 per byte of codes and gives one workgroup per
// (sequence, head) a 128-query tile that is mostly padding: 8 sequences of up
// to 4000 tokens, 32 heads, 5 queries took 213 us (staging 91, attention
// 124) for 102 MB of pages.
//
// Work: a workgroup of 4 waves owns 16 * QB queries of one (sequence, head)
// and one split of its visible 16-token chunks; a wave takes two chunks (32
// tokens) per step, steps dealt round-robin. Per step and wave:
//  * S^T = K Q^T on v_mfma_f32_16x16x32_f16, one chain per token half h: row
//    R of the A operand is token (R % 8) + 8 h of chunk R / 8, which is how a
//    page interleaves its tokens (lane 8p + c holds p and p + 8);
//  * lane (n, g) = (lane % 16, lane / 16) then holds for query n the scores
//    of rows 4g .. 4g + 3 in both halves: tokens p and p + 8 for p = 4 (g % 2)
//    .. + 3 of chunk g / 2. The same lane is column n, k-group g of the B
//    operand of O^T += V^T P^T, so with element 2 i + h = (p_i, half h) the
//    probabilities enter the second product without leaving their lane;
//  * an INT4 page's V word holds 4 dims of tokens p and p + 8, i.e. one
//    operand register (two k elements) for each of 4 output rows: unpacking
//    is the whole transpose. fp16 and token-major V are transposed with one
//    v_perm_b32 per register (fp16) or by unpacking two tokens together.
// Output row rr of V^T product i is dim (D / 16) rr + i.
//  * the loads of a step's K are issued when the previous step's K has been
//    used, those of V when its V has, the page lookups a step earlier;
//  * the softmax is the lazy running max of prefill.hip, per query column.
// Waves merge through LDS; splits write fp32 partials that direct_merge_kernel
// adds up (a launch of its own: the partials' workspace may hold anything).
#include <algorithm>
#include <cmath>

#include "attention.hpp"
#include "page_format.hpp"

namespace memopt {

typedef _Float16 half8d_t __attribute__((ext_vector_type(8)));
typedef float float4d_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4d_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2d_t __attribute__((ext_vector_type(2)));

struct DirectParams {
  const half_t *q;
  half_t *out;
  int32_t Lq, H, bs;
  const uint8_t *k, *v;       // code / element bases (INT4 pages: k = the page buffer)
  const void *ks, *vs;        // token-major scales
  int64_t kv_ps, kv_hs, kv_ts;  // bytes
  int64_t sc_ps, sc_hs, sc_ts;  // elements
  int32_t scale_f16;
  int64_t nb;
  const int32_t *bt;
  int32_t M;
  const int32_t *ctx;
  int32_t W, sinks, causal;
  float qk_scale_log2;
  int32_t splits;
  float *ws_o, *ws_ml;        // [B * H * Lq][splits][D], [B * H * Lq][splits][2]
};

// Output element from a query's weighted sum x and row sum l; 0 where no key
// was visible. Where a score is NaN or +inf (an inf or NaN key scale, a query
// that is not finite) l is NaN: over token-major codes the output is 0 then,
// as the generic kernel's and the oracle's; over pages and fp16 pools x is NaN
// and stays it, as on the staged path.
template <bool ROWS>
__device__ __forceinline__ half_t normalized(float x, float l) {
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;
  return ROWS && !(l > 0.0f) ? (half_t)0.0f : (half_t)(x * inv);
}

// Raw registers of one step, by cache format.
template <int D, int FMT>
struct DirectK;
template <int D>
struct DirectK<D, MEMOPT_KV_INT4> {
  uint32_t w[D / 16];  // kk-th operand word of half h: see k_word
  uint32_t sc;         // fp16 scales of (p, p + 8)
};
template <int D>
struct DirectK<D, MEMOPT_KV_INT4_ROWS> {
  uint32_t w[2][D / 32];
  float sc[2];
};
template <int D>
struct DirectK<D, MEMOPT_KV_FP16> {
  u32x4d_t w[2][D / 32];
};
template <int D, int FMT>
struct DirectV;
template <int D>
struct DirectV<D, MEMOPT_KV_INT4> {
  uint32_t w[4][D / 64];  // [p_i][unit]
  u32x4d_t sc;            // pair (p_i, p_i + 8) in word i
};
template <int D>
struct DirectV<D, MEMOPT_KV_INT4_ROWS> {
  uint32_t w[8];  // token e: D / 16 nibbles
  float sc[8];
};
template <int D>
struct DirectV<D, MEMOPT_KV_FP16> {
  uint32_t w[8][D / 32];  // token e: D / 16 halves
};

// fp16((code - 8) * s) of nibble `sh` (a bit offset) of w in two roundings,
// as the reference's dequantize kernel: the product in fp32, then fp16. The
// nibble becomes the float 2^23 + code by its bit pattern, exactly.
__device__ __forceinline__ half_t dequant_f32(uint32_t w, int sh, float s) {
  const float f = __uint_as_float(0x4B000000u | ((w >> sh) & 0xFu)) - 8388616.0f;
  return (half_t)__fmul_rn(f, s);
}

template <int D, int FMT, int QB>
__global__ __launch_bounds__(256, QB == 1 && (FMT == MEMOPT_KV_INT4 || D == 64) ? 3 : 2) void direct_kernel(
    const DirectParams p) {
  constexpr int NW = 4, KK = D / 32, ND = D / 16, QN = 16 * QB;
  constexpr bool PAGES = FMT == MEMOPT_KV_INT4, ROWS = FMT == MEMOPT_KV_INT4_ROWS;
  constexpr int OS = D + 4;  // row stride of s_o: 16 rows of D floats would share a bank
  __shared__ __attribute__((aligned(16))) float s_o[NW][QN][OS];
  __shared__ float s_ml[NW][QN][2];

  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int32_t split = blockIdx.x % p.splits, bh = blockIdx.x / p.splits;
  const int32_t h = bh % p.H, b = bh / p.H, q0 = blockIdx.y * QN;
  const int32_t ctx = p.ctx[b];
  const int32_t kv_lim = min(ctx, p.M * p.bs);
  const bool causal = p.causal != 0;
  const int32_t qlast = min(q0 + QN, p.Lq) - 1;
  const int32_t pos_lo = ctx - p.Lq + q0, pos_hi = ctx - p.Lq + qlast;

  // Visible chunks: sinks [0, sc), then the window [wc0, hc).
  const int32_t hi = max(0, causal ? min(kv_lim, pos_hi + 1) : kv_lim);
  const int32_t win_lo = max(0, causal ? pos_lo - p.W + 1 : ctx - p.W);
  const int32_t hc = (hi + 15) >> 4;
  const int32_t sc = (min(p.sinks, hi) + 15) >> 4;
  const int32_t wc0 = max(win_lo >> 4, sc);
  const int32_t n_vis = sc + max(0, hc - wc0);
  const SplitRange sr = split_range((n_vis + 1) >> 1, split, p.splits);
  const int32_t begin = sr.begin, end = sr.end;

  // Q as the B operand: column r = query, k-group g; dims of the kk-th
  // product as the K operand holds them (INT4: lane group g owns dims
  // [D/4 g, D/4 (g + 1)), pages in nibble-unpack order; fp16: 32 kk + 8 g).
  half8d_t qf[QB][KK];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int32_t qi = q0 + 16 * qb + r;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      half8d_t x = {};
      if (qi < p.Lq) {
        const int d0 = FMT == MEMOPT_KV_FP16 ? 32 * kk + 8 * g : (D / 4) * g + 8 * kk;
        const half8d_t n = __builtin_bit_cast(
            half8d_t, *reinterpret_cast<const u32x4d_t *>(p.q + (((int64_t)b * p.Lq + qi) * p.H + h) * D + d0));
        if (PAGES) {
          x[0] = n[0]; x[1] = n[4]; x[2] = n[1]; x[3] = n[5];
          x[4] = n[2]; x[5] = n[6]; x[6] = n[3]; x[7] = n[7];
        } else {
          x = n;
        }
      }
      qf[qb][kk] = x;
    }
  }

  float4d_t o[QB][ND];
  float ncm[QB], thr[QB], lsum[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
#pragma unroll
    for (int i = 0; i < ND; ++i) o[qb][i] = (float4d_t){};
    ncm[qb] = 0.0f;
    thr[qb] = -INFINITY;
    lsum[qb] = 0.0f;
  }

  // Chunk i of the visible list: logical chunk, and its offset from the
  // cache base (chunk 0 of page 0, always mapped, if there is none).
  struct Chunk {
    int32_t lc;
    bool ok;
    int64_t kv, sc;  // byte offset of its first token (this head), element offset of its scales
  };
  const int32_t *btrow = p.bt + (int64_t)b * p.M;
  const int32_t cpp = PAGES ? 1 : p.bs >> 4;
  const int32_t nb32 = (int32_t)min(p.nb, (int64_t)INT32_MAX);
  struct Entry {  // a chunk's block-table entry, not yet waited for
    int32_t lc, page, phys;
    bool in;
  };
  auto fetch = [&](int32_t i) __attribute__((always_inline)) {
    Entry e;
    e.lc = i < sc ? i : wc0 + (i - sc);
    e.in = i < n_vis;
    e.page = cpp == 1 ? e.lc : e.lc / cpp;
    e.phys = btrow[e.in ? e.page : 0];  // n_vis > 0 here, so the row has an entry 0
    return e;
  };
  auto resolve = [&](const Entry &e) __attribute__((always_inline)) {
    Chunk c;
    c.lc = e.lc;
    c.ok = e.in && e.phys >= 0 && e.phys < nb32;
    const int64_t pg = c.ok ? e.phys : 0;
    const int32_t pos = c.ok ? 16 * (e.lc - e.page * cpp) : 0;
    c.kv = pg * p.kv_ps + (int64_t)h * p.kv_hs + (int64_t)pos * p.kv_ts;
    c.sc = ROWS ? pg * p.sc_ps + (int64_t)h * p.sc_hs + (int64_t)pos * p.sc_ts : 0;
    return c;
  };

  const Int4Page f(D);
  DirectK<D, FMT> kr;
  DirectV<D, FMT> vr;
  auto scale_at = [&](const void *s, int64_t i) __attribute__((always_inline)) {
    return p.scale_f16 ? (float)reinterpret_cast<const half_t *>(s)[i] : reinterpret_cast<const float *>(s)[i];
  };
  // K of two chunks: lane row r is tokens r % 8 and r % 8 + 8 of chunk r / 8.
  auto load_k = [&](const Chunk &ca, const Chunk &cb) __attribute__((always_inline)) {
    const int pr = r & 7;
    const uint8_t *base = p.k + (r < 8 ? ca.kv : cb.kv);
    if constexpr (PAGES) {
      const u32x4d_t *src = reinterpret_cast<const u32x4d_t *>(base + f.kcodes + (8 * pr + 2 * g) * f.BPL);
#pragma unroll
      for (int i = 0; i < D / 64; ++i) {
        const u32x4d_t x = src[i];
#pragma unroll
        for (int j = 0; j < 4; ++j) kr.w[4 * i + j] = x[j];
      }
      kr.sc = *reinterpret_cast<const uint32_t *>(base + f.kscales + 2 * ((g * (D / 4) / 64) * 16 + 2 * pr));
    } else if constexpr (ROWS) {
      const int64_t sb = r < 8 ? ca.sc : cb.sc;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const uint8_t *src = base + (int64_t)(pr + 8 * t) * p.kv_ts + (D / 8) * g;
        if constexpr (D == 128) {
          const u32x4d_t x = *reinterpret_cast<const u32x4d_t *>(src);
#pragma unroll
          for (int j = 0; j < 4; ++j) kr.w[t][j] = x[j];
        } else {
          const u32x2d_t x = *reinterpret_cast<const u32x2d_t *>(src);
          kr.w[t][0] = x[0];
          kr.w[t][1] = x[1];
        }
        kr.sc[t] = scale_at(p.ks, sb + (int64_t)(pr + 8 * t) * p.sc_ts + g * (D / 4) / 64);
      }
    } else {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int kk = 0; kk < KK; ++kk)
          kr.w[t][kk] = *reinterpret_cast<const u32x4d_t *>(base + (int64_t)(pr + 8 * t) * p.kv_ts +
                                                            2 * (32 * kk + 8 * g));
    }
  };
  // V of two chunks: lane (r, g) holds dims [D/16 r, D/16 (r + 1)) of tokens
  // p_i, p_i + 8, p_i = 4 (g % 2) + i, of chunk g / 2 (element 2 i + t).
  auto load_v = [&](const Chunk &ca, const Chunk &cb) __attribute__((always_inline)) {
    const int p0 = 4 * (g & 1);
    const int64_t cbase = g < 2 ? ca.kv : cb.kv;
    if constexpr (PAGES) {
      const uint8_t *base = p.k + cbase;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint8_t *src = base + f.vcodes + 8 * (p0 + i) * f.BPL + (D / 16) * r;
        if constexpr (D == 128) {
          const u32x2d_t x = *reinterpret_cast<const u32x2d_t *>(src);
          vr.w[i][0] = x[0];
          vr.w[i][1] = x[1];
        } else {
          vr.w[i][0] = *reinterpret_cast<const uint32_t *>(src);
        }
      }
      vr.sc = *reinterpret_cast<const u32x4d_t *>(base + f.vscales + 2 * ((r * (D / 16) / 64) * 16 + 2 * p0));
    } else {
      const uint8_t *base = p.v + cbase;
      const int64_t sb = g < 2 ? ca.sc : cb.sc;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int t = p0 + (e >> 1) + 8 * (e & 1);
        if constexpr (ROWS) {
          const uint8_t *src = base + (int64_t)t * p.kv_ts + (D / 32) * r;
          if constexpr (D == 128) vr.w[e] = *reinterpret_cast<const uint32_t *>(src);
          else vr.w[e] = *reinterpret_cast<const uint16_t *>(src);
          vr.sc[e] = scale_at(p.vs, sb + (int64_t)t * p.sc_ts + r * (D / 16) / 64);
        } else {
          const uint8_t *src = base + (int64_t)t * p.kv_ts + (D / 8) * r;
          if constexpr (D == 128) {
            const u32x4d_t x = *reinterpret_cast<const u32x4d_t *>(src);
#pragma unroll
            for (int j = 0; j < 4; ++j) vr.w[e][j] = x[j];
          } else {
            const u32x2d_t x = *reinterpret_cast<const u32x2d_t *>(src);
            vr.w[e][0] = x[0];
            vr.w[e][1] = x[1];
          }
        }
      }
    }
  };

  const half2_t b1032 = {(half_t)1032.0f, (half_t)1032.0f}, b72 = {(half_t)72.0f, (half_t)72.0f};
  // The four half pairs of a page word, times s2 (exact codes, one rounding).
  auto unpack = [&](uint32_t w, half2_t s2) __attribute__((always_inline)) {
    const uint32_t w8 = w >> 8;
    return u32x4d_t{as_u32((as_half2(bfi(0x000F000Fu, w, 0x64006400u)) - b1032) * s2),
                    as_u32((as_half2(bfi(0x00F000F0u, w, 0x54005400u)) - b72) * s2),
                    as_u32((as_half2(bfi(0x000F000Fu, w8, 0x64006400u)) - b1032) * s2),
                    as_u32((as_half2(bfi(0x00F000F0u, w8, 0x54005400u)) - b72) * s2)};
  };
  // K operand of product kk, token half t.
  auto k_operand = [&](int t, int kk) __attribute__((always_inline)) {
    if constexpr (PAGES) {
      const half2_t s = as_half2(kr.sc);
      const half2_t s2 = t ? half2_t{s.y, s.y} : half2_t{s.x, s.x};
      const uint32_t w = D == 128 ? kr.w[4 * (kk >> 1) + 2 * t + (kk & 1)] : kr.w[2 * kk + t];
      return __builtin_bit_cast(half8d_t, unpack(w, s2));
    } else if constexpr (ROWS) {
      half8d_t x;
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = dequant_f32(kr.w[t][kk], 4 * e, kr.sc[t]);
      return x;
    } else {
      return __builtin_bit_cast(half8d_t, kr.w[t][kk]);
    }
  };

  // 8 |scale| past the fp16 range (or NaN): a code may dequantize to inf or NaN.
  auto odd_scale = [](float x) { return (__float_as_uint(x) & 0x7FFFFFFFu) > 0x45FFC000u; };  // 8184
  bool odd_v = false;
  const half2_t ones = {(half_t)1.0f, (half_t)1.0f};
  // exp2 argument of a new maximum: probabilities lie in (0, 2^15], so fp16
  // holds those down to 2^-21 of the largest as normal numbers.
  constexpr float kTop = 7.0f;
  auto step = [&](const Chunk &ca, const Chunk &cb, const Chunk &na, const Chunk &nb_, bool more)
                  __attribute__((always_inline)) {
    float4d_t s[QB][2];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const half8d_t a = k_operand(t, kk);
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
          s[qb][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, qf[qb][kk], kk == 0 ? (float4d_t){} : s[qb][t], 0, 0, 0);
      }
    }
    if (more) load_k(na, nb_);

    // Every (token, query) of the step visible: no mask (wave-uniform).
    const int32_t ta = ca.lc * 16, tb = cb.lc * 16;
    auto chunk_full = [&](const Chunk &c, int32_t t0) {
      const bool seen = causal ? t0 + 15 <= pos_lo && (t0 >= pos_hi - p.W + 1 || t0 + 16 <= p.sinks)
                               : t0 >= ctx - p.W || t0 + 16 <= p.sinks;
      return c.ok && t0 + 16 <= kv_lim && seen;
    };
    const bool full = chunk_full(ca, ta) && chunk_full(cb, tb);
    const int32_t key0 = (g < 2 ? ta : tb) + 4 * (g & 1);
    const bool c_ok = g < 2 ? ca.ok : cb.ok;
    half8d_t pf[QB], pl[ROWS ? QB : 1];
    // Token-major codes: the probabilities keep about 22 bits as the sum of
    // two fp16 operands (with one, the error against 64 bits was 2.3e-4 where
    // a softmax in fp32 has 2.1e-4). V elements that are not finite must not
    // meet the second operand's zeros, nor the probability 0 of a query that
    // does not see their token: scales that may make one count as 0 here, and
    // their tokens are added after the last step.
    if constexpr (ROWS) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const bool odd = odd_scale(vr.sc[e]);
        odd_v |= odd;
        vr.sc[e] = odd ? 0.0f : vr.sc[e];
      }
    }
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      float x[8];  // element 2 i + t: token key0 + i + 8 t
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = fmaf(s[qb][e & 1][e >> 1], p.qk_scale_log2, ncm[qb]);
      if (!full) {
        // (bounds relative to the lane's first key, one test per element and
        // no branch: as short-circuited conditions a masked step took about
        // 1200 instructions more than a full one)
        const int32_t pos = ctx - p.Lq + q0 + 16 * qb + r;
        const int32_t last = c_ok ? (causal ? min(pos, kv_lim - 1) : kv_lim - 1) - key0 : -1;
        const int32_t first_w = (causal ? pos - p.W + 1 : ctx - p.W) - key0, end_s = p.sinks - key0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int32_t c = (e >> 1) + 8 * (e & 1);
          const bool vis = (c <= last) & ((c >= first_w) | (c < end_s));
          x[e] = vis ? x[e] : -INFINITY;
        }
      }
      float t = x[0];
#pragma unroll
      for (int e = 1; e < 8; ++e) t = fmaxf(t, x[e]);
      if (__any(t > thr[qb])) {  // wave-uniform, rare after the first steps
        // the query's four lanes agree on the new maximum
        auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(t), __float_as_uint(t), false, false);
        t = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
        sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(t), __float_as_uint(t), false, false);
        t = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
        const bool first = thr[qb] == -INFINITY, found = t > -INFINITY;
        const float shift = first ? (found ? t - kTop : 0.0f) : fmaxf(t - kTop, 0.0f);
        const float alpha = first ? (found ? 0.0f : 1.0f) : (shift > 0.0f ? fast_exp2(-shift) : 1.0f);
        lsum[qb] *= alpha;
#pragma unroll
        for (int i = 0; i < ND; ++i) o[qb][i] *= alpha;
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] -= shift;
        ncm[qb] -= shift;
        thr[qb] = (first && !found) ? thr[qb] : kTop + 8.0f;
      }
      uint32_t w[4];
      if constexpr (ROWS) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float pe = fast_exp2(x[e]);
          lsum[qb] += pe;
          pf[qb][e] = (half_t)pe;
          pl[qb][e] = (half_t)(pe - (float)pf[qb][e]);
        }
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          w[i] = as_u32(half2_t{(half_t)fast_exp2(x[2 * i]), (half_t)fast_exp2(x[2 * i + 1])});
          lsum[qb] = __builtin_amdgcn_fdot2(as_half2(w[i]), ones, lsum[qb], false);
        }
        pf[qb] = __builtin_bit_cast(half8d_t, u32x4d_t{w[0], w[1], w[2], w[3]});
      }
    }

    // V of tokens past the context or without a page may hold any bits; it
    // becomes zero, as P = 0 must not meet NaN.
    if (!full) {
      const int32_t live_c = c_ok ? kv_lim - key0 : 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const bool live = (e >> 1) + 8 * (e & 1) < live_c;
        if constexpr (PAGES) {
          vr.sc[e >> 1] &= live ? ~0u : (e & 1) ? 0x0000FFFFu : 0xFFFF0000u;
        } else if constexpr (ROWS) {
          vr.sc[e] = live ? vr.sc[e] : 0.0f;
        } else {
#pragma unroll
          for (int j = 0; j < D / 32; ++j) vr.w[e][j] = live ? vr.w[e][j] : 0u;
        }
      }
    }
    auto pv = [&](int i, u32x4d_t a) __attribute__((always_inline)) {
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        o[qb][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8d_t, a), pf[qb], o[qb][i], 0, 0, 0);
        if constexpr (ROWS)
          o[qb][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8d_t, a), pl[qb], o[qb][i], 0, 0, 0);
      }
    };
    if constexpr (PAGES) {
#pragma unroll
      for (int u = 0; u < D / 64; ++u) {
        u32x4d_t x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = unpack(vr.w[i][u], as_half2(vr.sc[i]));
#pragma unroll
        for (int j = 0; j < 4; ++j) pv(4 * u + j, u32x4d_t{x[0][j], x[1][j], x[2][j], x[3][j]});
      }
    } else if constexpr (ROWS) {
#pragma unroll
      for (int i = 0; i < ND; ++i) {
        u32x4d_t a;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          a[j] = as_u32(half2_t{dequant_f32(vr.w[2 * j], 4 * i, vr.sc[2 * j]),
                                dequant_f32(vr.w[2 * j + 1], 4 * i, vr.sc[2 * j + 1])});
        pv(i, a);
      }
    } else {
#pragma unroll
      for (int i = 0; i < ND; ++i) {
        u32x4d_t a;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          a[j] = __builtin_amdgcn_perm(vr.w[2 * j + 1][i >> 1], vr.w[2 * j][i >> 1], (i & 1) ? 0x07060302u : 0x05040100u);
        pv(i, a);
      }
    }
    if (more) load_v(na, nb_);
  };

  int32_t st = begin + wave;
  if (st < end) {
    Entry ea = fetch(2 * (st + NW)), eb = fetch(2 * (st + NW) + 1);
    Chunk ca = resolve(fetch(2 * st)), cb = resolve(fetch(2 * st + 1));
    load_k(ca, cb);
    load_v(ca, cb);
    for (; st < end; st += NW) {
      const Chunk na = resolve(ea), nb_ = resolve(eb);
      ea = fetch(2 * (st + 2 * NW));
      eb = fetch(2 * (st + 2 * NW) + 1);
      step(ca, cb, na, nb_, st + NW < end);
      ca = na;
      cb = nb_;
    }
  }

  if constexpr (ROWS) {
    if (__any(odd_v)) {
      // Token by token: each lane takes the score over its quarter of the
      // dims, and adds its quarter of V (the row sums have the token already).
#pragma unroll 1
      for (int32_t i = 2 * (begin + wave); i < 2 * end; i += (i & 1) ? 2 * NW - 1 : 1) {
        const Chunk c = resolve(fetch(i));
#pragma unroll 1
        for (int t = 0; t < 16 && c.ok; ++t) {
          const int32_t key = c.lc * 16 + t;
          if (key >= kv_lim) break;
          const int64_t si = c.sc + (int64_t)t * p.sc_ts + g * (D / 4) / 64;
          const float vs = scale_at(p.vs, si);
          if (!__any(odd_scale(vs))) continue;
          const float ks = scale_at(p.ks, si);
          const uint8_t *krow = p.k + c.kv + (int64_t)t * p.kv_ts + (D / 8) * g;
          const uint8_t *vrow = p.v + c.kv + (int64_t)t * p.kv_ts + (D / 8) * g;
#pragma unroll
          for (int qb = 0; qb < QB; ++qb) {
            float s = 0.0f;
#pragma unroll
            for (int d = 0; d < D / 4; ++d)
              s = fmaf((float)qf[qb][d >> 3][d & 7], (float)dequant_f32(krow[d >> 1], 4 * (d & 1), ks), s);
            s = xor32_sum(xor16_sum(s));
            const int32_t pos = ctx - p.Lq + q0 + 16 * qb + r;
            const bool vis = causal ? key <= pos && (key < p.sinks || key >= pos - p.W + 1)
                                    : key >= ctx - p.W || key < p.sinks;
            const float pe = fast_exp2(fmaf(s, p.qk_scale_log2, ncm[qb]));
            if (vis && odd_scale(vs)) {
#pragma unroll
              for (int d = 0; d < D / 4; ++d)
                o[qb][d % ND][d / ND] =
                    fmaf(pe, (float)dequant_f32(vrow[d >> 1], 4 * (d & 1), vs), o[qb][d % ND][d / ND]);
            }
          }
        }
      }
    }
  }

  // Merge of the waves. Lane (n, g) holds dims [D/4 g, D/4 (g + 1)) of query
  // n: row 4 g + reg of V^T product i is dim D/16 (4 g + reg) + i.
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const float l = xor32_sum(xor16_sum(lsum[qb]));
    const int row = 16 * qb + r;
#pragma unroll
    for (int reg = 0; reg < 4; ++reg)
#pragma unroll
      for (int i = 0; i < ND; i += 4)
        *reinterpret_cast<float4d_t *>(&s_o[wave][row][ND * (4 * g + reg) + i]) =
            float4d_t{o[qb][i][reg], o[qb][i + 1][reg], o[qb][i + 2][reg], o[qb][i + 3][reg]};
    if (g == 0) {
      s_ml[wave][row][0] = thr[qb] == -INFINITY ? -INFINITY : -ncm[qb];
      s_ml[wave][row][1] = l;
    }
  }
  __syncthreads();
  for (int idx = tid; idx < QN * (D / 4); idx += NW * 64) {
    const int row = idx / (D / 4), d = 4 * (idx % (D / 4));
    const int32_t qi = q0 + row;
    if (qi >= p.Lq) break;  // rows grow with idx
    float mx = s_ml[0][row][0];
#pragma unroll
    for (int w = 1; w < NW; ++w) mx = fmaxf(mx, s_ml[w][row][0]);
    float l = 0.0f;
    float4d_t x = {};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float mw = s_ml[w][row][0], fw = mw == -INFINITY ? 0.0f : fast_exp2(mw - mx);
      l += s_ml[w][row][1] * fw;
      x += *reinterpret_cast<const float4d_t *>(&s_o[w][row][d]) * fw;
    }
    const int64_t qrow = ((int64_t)b * p.H + h) * p.Lq + qi;
    if (p.splits == 1) {
      const half2_t y0 = {normalized<ROWS>(x[0], l), normalized<ROWS>(x[1], l)};
      const half2_t y1 = {normalized<ROWS>(x[2], l), normalized<ROWS>(x[3], l)};
      *reinterpret_cast<u32x2d_t *>(p.out + (((int64_t)b * p.Lq + qi) * p.H + h) * D + d) =
          u32x2d_t{as_u32(y0), as_u32(y1)};
    } else {
      const int64_t slot = qrow * p.splits + split;
      *reinterpret_cast<float4d_t *>(p.ws_o + slot * D + d) = x;
      if (d == 0) {
        p.ws_ml[2 * slot] = mx;
        p.ws_ml[2 * slot + 1] = l;
      }
    }
  }
}

// Sums the splits of one query row, one wave per row: lane s takes split s's
// (m, l) (splits <= 64); every lane then adds D / 64 dims over the splits,
// eight loads in flight.
template <int D, bool ROWS>
__global__ __launch_bounds__(256) void direct_merge_kernel(const DirectParams p, int64_t rows) {
  constexpr int R = 8, E = D / 64;
  typedef float vec_t __attribute__((ext_vector_type(E)));
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (row >= rows) return;
  const float *ml = p.ws_ml + 2 * (row * p.splits + min(lane, p.splits - 1));
  const float *src = p.ws_o + row * p.splits * D + E * lane;
  const float m = lane < p.splits ? ml[0] : -INFINITY, l = ml[1];
  const float mx = wave_max(m);
  const float wgt = m == -INFINITY ? 0.0f : fast_exp2(m - mx);
  float lt = lane < p.splits ? l * wgt : 0.0f;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) lt += shfl_xor(lt, off);
  vec_t o = {};
  for (int s0 = 0; s0 < p.splits; s0 += R) {
    vec_t x[R];
#pragma unroll
    for (int k = 0; k < R; ++k)
      x[k] = *reinterpret_cast<const vec_t *>(src + (int64_t)min(s0 + k, p.splits - 1) * D);
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const float fs = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(wgt), min(s0 + k, 63)));
      if (s0 + k < p.splits) o += x[k] * fs;
    }
  }
  const int32_t qi = (int32_t)(row % p.Lq);
  const int64_t bh = row / p.Lq, h = bh % p.H, b = bh / p.H;
  half_t *dst = p.out + ((b * p.Lq + qi) * p.H + h) * D + E * lane;
  if constexpr (E == 2) *reinterpret_cast<uint32_t *>(dst) = as_u32(half2_t{normalized<ROWS>(o[0], lt), normalized<ROWS>(o[1], lt)});
  else *dst = normalized<ROWS>(o[0], lt);
}

// Query blocks of 16 * QB rows: two blocks of 16 share every K and V operand
// once there are more than 16 queries.
static int direct_qb(const memopt_attn_desc &d) { return d.q_len <= 16 ? 1 : 2; }

// Where the direct kernel beats the staged path (staging and attention
// launches together). Both times are estimated, in us, from sums fitted to
// both paths timed on 96000 random calls over pages and fp16 pools (1 to 40
// heads, 1 to 16 sequences, 2 to 8192 queries, 20 to 32768 tokens, windows,
// causal or not, equal and unequal lengths; median error 4 to 6 %):
//  * a workgroup takes a fixed time and one per key it visits, and `both`
//    more of that when a second one shares its CU; past two per CU the grid
//    runs in rounds, whose last one counts `ramp` in full (causal staged
//    grids start their longest tiles first, which fills it);
//  * a causal staged grid ends with its longest tile;
//  * staging a (token, head, dim) of K and V costs `stage` per million;
//  * each block of 32 queries reads its keys again: from 256 heads on these
//    reads leave the caches, at about 7 TB/s (16 sequences of 2277 fp16 tokens
//    x 32 heads of 128, 486 queries: 1571 us, staged 576).
// The estimates decide above 128 queries and 128 tiles (fewer tiles leave half
// of the CUs idle on the staged path). Fixed numbers of queries, tiles and
// (query, key) pairs, which drew the line before, lost 8 to 45 % on 266 of
// 61500 calls (4 x 4 heads of 128, 3540 queries in a 512-token window, not
// causal: 50 us, staged 40; 1 x 32 heads, fp16, 1687 causal queries: 51 and
// 44; 2 x 40 heads, 530 queries: 49 and 43). On 31300 further random calls
// this rule takes a path more than 8 % slower than the staged one 41 times,
// and one more than 15 % slower than the better one 97 times.
struct PathCost {
  double block, key, both;       // direct: per block, per thousand keys
  double tile, tile_key, tile_both, stage;
};
static const PathCost kPathCost[2][2] = {
    // D = 64, 128
    {{1.3, 6.2, 0.37, 2.4, 21.0, 0.285, 0.94}, {2.7, 7.3, 0.85, 6.4, 24.6, 0.42, 0.76}},   // pages
    {{1.3, 7.3, 0.46, 2.4, 21.0, 0.285, 1.33}, {1.95, 8.1, 1.18, 6.4, 24.6, 0.42, 1.01}},  // fp16 pools
};

// Time of n equal workgroups in units of one alone on its CU.
static double grid_time(double n, double both, double ramp) {
  const double x = n / compute_units(), fill = 1.0 + both * std::min(1.0, std::max(0.0, x - 1.0));
  return fill * (x <= 2.0 ? 1.0 : (1.0 - ramp) * x / 2 + ramp * std::ceil(x / 2));
}

// (An environment variable in its place cost each call 1 us.)
static thread_local int32_t t_path = MEMOPT_PATH_AUTO;

static bool direct_faster(const memopt_attn_desc &d) {
  if (t_path != MEMOPT_PATH_AUTO) return t_path == MEMOPT_PATH_DIRECT;
  const int64_t q = d.q_len, heads = (int64_t)d.num_heads * d.batch, tiles = (q + 127) / 128 * heads;
  if (q <= 128 || tiles <= 128) return true;
  // Pairs of one sequence at the longest context the block table holds.
  const int64_t T = (int64_t)d.max_blocks_per_seq * d.block_size;
  const int64_t W = std::min<int64_t>(effective_window(d.window_size, d.max_seq_len), T);
  int64_t pairs = q * W;
  if (d.causal) {  // sum of min(W, pos + 1) over the query positions T - q .. T - 1
    const int64_t lo = std::max<int64_t>(0, T - q), full = std::max(lo, std::min(W, T));
    pairs = (full - lo) * (full + lo + 1) / 2 + (T - full) * W;
  }
  const bool pages = d.kv_format == MEMOPT_KV_INT4, clip = W < T, sinks = clip && d.num_sink_tokens > 0;
  const PathCost &c = kPathCost[pages ? 0 : 1][d.head_dim == 128];
  // Thousands of keys a block or tile visits, ragged edges included.
  const double mean = (double)pairs / (double)q;
  const double keys = 1e-3 * (mean + (!d.causal ? 0 : clip ? 24 : 8) + (sinks ? 16 : 0));
  const double tile_keys = 1e-3 * (mean + (!d.causal ? 0 : clip ? 96 : 32) + (sinks ? 64 : 0));
  const double longest = 1e-3 * (double)(d.causal ? std::min(T, W + 127) : W);
  const double blocks = (double)((q + 31) / 32);
  const double melems = 1e-6 * (double)(std::min(T, d.causal ? q + W : W) * heads * d.head_dim);  // K and V staged
  const double staged = 10.0 + 17.7 * (longest - tile_keys) + c.stage * melems +
                        (c.tile + c.tile_key * tile_keys) *
                            grid_time((double)tiles, c.tile_both, d.causal ? 0.08 : 0.65);
  const double compute = 4.5 + (c.block + c.key * keys) * grid_time(blocks * heads, c.both, 0.42);
  // MB that the blocks of all heads read at once, and how often
  const double mb = 1e-3 * keys * heads * d.head_dim * (pages ? 1.125 : 4.0);
  const double passes = blocks * std::min(1.0, heads / 256.0);
  const double direct = std::max(compute, passes > 1.0 ? passes * mb / 7.0 : 0.0);
  return direct < 0.95 * staged;
}

static int64_t direct_query_blocks(const memopt_attn_desc &d) {
  const int64_t qn = 16 * direct_qb(d);
  return (d.q_len + qn - 1) / qn;
}

bool direct_supported(const memopt_attn_desc &d) {
  if (direct_query_blocks(d) > 65535) return false;  // a grid dimension
  auto al = [](const void *x, int64_t a) { return ((uintptr_t)x & (uintptr_t)(a - 1)) == 0; };
  if (d.q_len < 2 || (d.head_dim != 64 && d.head_dim != 128) || d.num_kv_blocks <= 0) return false;
  if (!al(d.query, 16) || !al(d.out, 16)) return false;
  if (d.kv_format != MEMOPT_KV_INT4_ROWS) return prefill_supported(d) && direct_faster(d);
  if (d.block_size % 16 != 0) return false;
  // 16-byte (D = 128) or 8-byte loads of a token's codes
  const int64_t a = d.head_dim / 8;
  return al(d.key_cache, a) && al(d.value_cache, a) && d.kv_page_stride % a == 0 && d.kv_head_stride % a == 0 &&
         d.kv_token_stride % a == 0;
}

// Splits of a call: about two workgroups per CU (three or more: 12 % slower at
// 16 sequences of 2000 fp16 tokens, 30 % at 64 queries of one sequence), at least two steps (64
// tokens) per wave, at most 64, and no more than `bytes` of partials hold
// (none without a workspace). Over INT4 pages and fp16 pools the partials are
// also no larger than the staged path's copy of K and V: with about as many
// queries as keys, writing and merging them costs more than the idle CUs
// (causal, 8 heads of 128, 1024 queries on 1024 tokens 17 us unsplit, 23 in 2
// splits; 800 on 800 over fp16 15 and 24 in 3; 12 heads of 64, 512 on 512 9
// and 13; with one or two heads they break even: 1100 on 1100 17 and 13 in 4,
// 2 x 2000 on 2000 26 and 25). Both entry points and the workspace query
// count by this rule, so they run the same splits wherever these fit.
static int32_t direct_splits(const memopt_attn_desc &d, int64_t bytes) {
  if (d.kv_format != MEMOPT_KV_INT4_ROWS) bytes = std::min(bytes, staged_copy_bytes(d));
  const int64_t rows = (int64_t)d.batch * d.num_heads * d.q_len;
  const int64_t qn = 16 * direct_qb(d);
  const int64_t wgs = (int64_t)d.batch * d.num_heads * direct_query_blocks(d);
  const int64_t W = effective_window(d.window_size, d.max_seq_len);
  const int64_t sinks = d.num_sink_tokens > 0 ? d.num_sink_tokens : 0;
  int64_t tokens = (d.causal ? W + qn : W) + sinks + 32;
  tokens = std::min<int64_t>(tokens, (int64_t)d.max_blocks_per_seq * d.block_size);
  int64_t s = (2LL * compute_units() + wgs - 1) / wgs;
  s = std::min(s, tokens / (4 * 2 * 32));
  s = std::min<int64_t>(s, 64);
  s = std::min(s, bytes / (rows * (d.head_dim + 2) * 4));
  return (int32_t)(s < 2 ? 1 : s);
}

int64_t direct_workspace_bytes(const memopt_attn_desc &d) {
  const int64_t s = direct_splits(d, INT64_MAX);
  return s > 1 ? (int64_t)d.batch * d.num_heads * d.q_len * s * (d.head_dim + 2) * 4 : 0;
}

template <int D, int FMT>
static void launch_direct_qb(const DirectParams &p, int qb, dim3 grid, hipStream_t stream) {
  if (qb == 1) hipLaunchKernelGGL((direct_kernel<D, FMT, 1>), grid, dim3(256), 0, stream, p);
  else hipLaunchKernelGGL((direct_kernel<D, FMT, 2>), grid, dim3(256), 0, stream, p);
}

int launch_direct(const memopt_attn_desc &d, int32_t W, float qk_scale_log2, hipStream_t stream) {
  DirectParams p = {};
  p.q = (const half_t *)d.query;
  p.out = (half_t *)d.out;
  p.Lq = d.q_len;
  p.H = d.num_heads;
  p.bs = d.block_size;
  p.k = (const uint8_t *)d.key_cache;
  p.v = (const uint8_t *)d.value_cache;
  if (d.kv_format == MEMOPT_KV_INT4) {
    const Int4Page f(d.head_dim);
    p.kv_ps = d.num_heads * f.block;
    p.kv_hs = f.block;
  } else {
    const int64_t eb = d.kv_format == MEMOPT_KV_FP16 ? 2 : 1;
    p.kv_ps = d.kv_page_stride * eb;
    p.kv_hs = d.kv_head_stride * eb;
    p.kv_ts = d.kv_token_stride * eb;
    p.ks = d.key_scales;
    p.vs = d.value_scales;
    p.sc_ps = d.sc_page_stride;
    p.sc_hs = d.sc_head_stride;
    p.sc_ts = d.sc_token_stride;
    p.scale_f16 = d.scale_dtype == MEMOPT_SCALE_F16;
  }
  p.nb = d.num_kv_blocks;
  p.bt = d.block_tables;
  p.M = d.max_blocks_per_seq;
  p.ctx = d.context_lens;
  p.W = std::min(W, 1 << 30);  // (so that position - W stays in 32 bits for positions below 0)
  p.sinks = d.num_sink_tokens < 0 ? 0 : d.num_sink_tokens;
  p.causal = d.causal;
  p.qk_scale_log2 = qk_scale_log2;
  p.splits = direct_splits(d, d.workspace ? d.workspace_bytes : 0);
  const int64_t rows = (int64_t)d.batch * d.num_heads * d.q_len;
  if (p.splits > 1) {
    p.ws_o = (float *)d.workspace;
    p.ws_ml = p.ws_o + rows * p.splits * d.head_dim;
  }
  const int qb = direct_qb(d);
  const int64_t gx = (int64_t)d.batch * d.num_heads * p.splits;
  MEMOPT_REQUIRE(gx < (1LL << 31), MEMOPT_ERR_UNSUPPORTED, "paged_attention: too many query blocks");
  const dim3 grid((unsigned)gx, (unsigned)direct_query_blocks(d));
  if (d.head_dim == 128) {
    if (d.kv_format == MEMOPT_KV_INT4) launch_direct_qb<128, MEMOPT_KV_INT4>(p, qb, grid, stream);
    else if (d.kv_format == MEMOPT_KV_FP16) launch_direct_qb<128, MEMOPT_KV_FP16>(p, qb, grid, stream);
    else launch_direct_qb<128, MEMOPT_KV_INT4_ROWS>(p, qb, grid, stream);
  } else {
    if (d.kv_format == MEMOPT_KV_INT4) launch_direct_qb<64, MEMOPT_KV_INT4>(p, qb, grid, stream);
    else if (d.kv_format == MEMOPT_KV_FP16) launch_direct_qb<64, MEMOPT_KV_FP16>(p, qb, grid, stream);
    else launch_direct_qb<64, MEMOPT_KV_INT4_ROWS>(p, qb, grid, stream);
  }
  int rc = check_launch("paged_attention(direct)");
  if (rc != MEMOPT_OK || p.splits == 1) return rc;
  const dim3 mgrid((unsigned)((rows + 3) / 4));
  const bool token_major = d.kv_format == MEMOPT_KV_INT4_ROWS;
  if (d.head_dim == 128) {
    if (token_major) hipLaunchKernelGGL((direct_merge_kernel<128, true>), mgrid, dim3(256), 0, stream, p, rows);
    else hipLaunchKernelGGL((direct_merge_kernel<128, false>), mgrid, dim3(256), 0, stream, p, rows);
  } else {
    if (token_major) hipLaunchKernelGGL((direct_merge_kernel<64, true>), mgrid, dim3(256), 0, stream, p, rows);
    else hipLaunchKernelGGL((direct_merge_kernel<64, false>), mgrid, dim3(256), 0, stream, p, rows);
  }
  return check_launch("paged_attention(direct merge)");
}

}  // namespace memopt

using namespace memopt;

extern "C" int memopt_multi_query_path(int32_t path) {
  MEMOPT_REQUIRE(path == MEMOPT_PATH_AUTO || path == MEMOPT_PATH_STAGED || path == MEMOPT_PATH_DIRECT,
                 MEMOPT_ERR_INVALID, "multi_query_path: unknown path");
  t_path = path;
  return MEMOPT_OK;
}
