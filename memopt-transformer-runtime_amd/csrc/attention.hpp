// attention.hpp — shared declarations of the paged-attention kernels.
#pragma once
#include "common.hpp"

namespace memopt {

// Key-visibility rule of one query, resolved to two token ranges:
// sinks [0, sink_end) and the window [win_lo, hi) (win_lo >= sink_end when
// the ranges are disjoint; they may overlap, the union is what counts).
struct KeyRange {
  int32_t sink_end, win_lo, hi;
};

// Non-causal (reference dynamic_sparse_attention, src/csrc/attention.cu:158-186,
// plus sinks): every query sees [max(0, ctx-W), ctx) U [0, min(sinks, ctx)).
// Causal (scripts/bench_accuracy.py:271-275): query at absolute position
// pos sees j <= pos && (j < sinks || j >= pos - W + 1).
__host__ __device__ inline KeyRange key_range(int32_t ctx, int32_t pos, int32_t W, int32_t sinks,
                                               bool causal) {
  KeyRange r;
  r.hi = causal ? (pos + 1 < ctx ? pos + 1 : ctx) : ctx;
  if (r.hi < 0) r.hi = 0;
  const int32_t top = causal ? pos + 1 : ctx;  // window anchored at pos (causal) or ctx
  r.win_lo = top - W;
  if (r.win_lo < 0) r.win_lo = 0;
  r.sink_end = sinks < r.hi ? sinks : r.hi;
  if (r.sink_end < 0) r.sink_end = 0;
  return r;
}

// Window of the reference signature: W <= 0 or W > max_seq_len means
// max_seq_len (src/csrc/attention.cu:453-455).
inline int32_t effective_window(int32_t window, int32_t max_seq_len) {
  return (window <= 0 || window > max_seq_len) ? max_seq_len : window;
}

// Visible pages (or 16-token chunks) [begin, end) of split `split` of
// `splits` over n of them, in 32-bit arithmetic: a 64-bit division expands
// to a long scalar sequence that sits on every decode launch's critical path.
struct SplitRange {
  int32_t begin, end;
};
__device__ __forceinline__ SplitRange split_range(int32_t n, int32_t split, int32_t splits) {
  if (splits <= 1) return {0, n};
  const int32_t q = n / splits, r = n - q * splits;
  const int32_t begin = split * q + (split < r ? split : r);
  return {begin, begin + q + (split < r ? 1 : 0)};
}

struct DecodeParams {
  const half_t *q;
  half_t *out;
  const uint8_t *kc, *vc;
  const void *ks, *vs;
  int64_t kv_ps, kv_hs, kv_ts;  // code strides, bytes
  int64_t sc_ps, sc_hs, sc_ts;  // scale strides, elements
  const int32_t *bt;
  const int32_t *ctx;
  int64_t nb;                   // pages in the pool (entries >= nb are skipped)
  int32_t pages;                // 1: this build's INT4 page format (page_format.hpp)
  int32_t M, H, W, sinks, splits;
  int32_t bs;           // tokens per page (fp16 pools; a multiple of 16)
  int32_t B, hc, groups;  // token-major codes: sequences, heads per cluster (1: grid order), clusters per sequence
  float qk_scale_log2;  // (1/sqrt(D)) * log2(e)
  float *ws_o;          // [B, H, splits, D] (splits > 1)
  float *ws_ml;         // [B, H, splits, 2]
  unsigned long long *ws_cnt;  // [B, H] arrival counters (splits > 1)
  unsigned long long tag;      // this launch's id, 1 .. 2^56 - 1
};

// Bytes of a decode call's split-K workspace: partials (o[D], m, l) per
// (b, h, split) and one arrival counter per (b, h).
inline int64_t decode_workspace_bytes(int64_t batch, int64_t heads, int64_t splits, int64_t D) {
  return splits > 1 ? batch * heads * (splits * (D + 2) * 4 + 8) : 0;
}

// Id of the next decode launch (for the arrival counters).
unsigned long long next_decode_tag();

// Epilogue of a decode workgroup of NW waves over (b, h, split): merges the
// waves' (m, l, acc[D]) held in LDS. Unsplit: writes the output row. Split:
// writes this split's partial to the workspace with agent-scope stores
// (they bypass the per-XCD L2s, as the splits of one (b, h) run on
// different XCDs), waits for them, and counts its arrival on (b, h) in a
// counter word tag << 8 | count: an atomic max with tag << 8 turns whatever
// an earlier launch left (smaller tags; zero at first) into count 0 and the
// add after it counts, one round trip and no retry. (A compare-and-swap per
// arrival, retried whenever another split got in between, cost about 2 us
// per split: one sequence of 131072 tokens x 32 heads in 24 splits took
// 146 us, with the add 97 us.) Two cases start elsewhere: a word above this
// tag (an older launch replayed from a graph after newer ones, or foreign
// data) is replaced by compare-and-swap, and a replay of the launch that
// used the word last starts at the full count and ends at twice that, from
// where the last split takes it back. A workspace zeroed once needs no
// clearing between launches (a fresh one must be zero: a stale word with
// this launch's tag would miscount). The split that completes the count
// merges every partial (log-sum-exp, agent-scope loads) into the output
// row. No workgroup waits for another.
template <int D, int NW>
__device__ __forceinline__ void decode_epilogue(const DecodeParams &p, int64_t bh, int32_t split,
                                                float (*s_acc)[D], const float (*s_ml)[2]) {
  for (int d = threadIdx.x; d < D; d += NW * 64) {
    float mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) mx = fmaxf(mx, s_ml[w][0]);
    float lt = 0.0f, o = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = (s_ml[w][0] == -INFINITY) ? 0.0f : fast_exp2(s_ml[w][0] - mx);
      lt += s_ml[w][1] * f;
      o += s_acc[w][d] * f;
    }
    if (p.splits == 1) {
      p.out[bh * D + d] = (half_t)(lt > 0.0f ? o / lt : 0.0f);
    } else {
      const int64_t slot = bh * p.splits + split;
      __hip_atomic_store(&p.ws_o[slot * D + d], o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (d == 0) {
        __hip_atomic_store(&p.ws_ml[slot * 2], mx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&p.ws_ml[slot * 2 + 1], lt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  if (p.splits == 1) return;
  __shared__ int s_last;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's partial stores are complete
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long *cnt = p.ws_cnt + bh, base = p.tag << 8;
    // (two operations of one lane on one address: they take effect in order)
    __hip_atomic_fetch_max(cnt, base, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    unsigned long long nv = __hip_atomic_fetch_add(cnt, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
    if (((nv - 1) >> 8) != p.tag) {  // a larger word was there
      unsigned long long e = __hip_atomic_load(cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      do {
        nv = (e >> 8) == p.tag ? e + 1 : base | 1;
      } while (!__hip_atomic_compare_exchange_strong(cnt, &e, nv, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT));
    }
    const int n = (int)(nv & 0xFF);
    s_last = n == p.splits || n == 2 * p.splits;
    if (n == 2 * p.splits)
      __hip_atomic_store(cnt, base | (unsigned)p.splits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!s_last) return;
  // The merge is two memory round trips, not two per split: every wave loads
  // all (m, l) pairs at once (lane s takes split s; splits <= 64), and the
  // o rows are dealt to NT / D parts of the workgroup, each with its loads
  // issued together before any is used, the parts' sums meeting in LDS.
  constexpr int NT = NW * 64, PARTS = NT / D, WPD = D / 64, R = 8;
  static_assert(NT % D == 0 && PARTS <= NW, "whole parts; their sums fit s_acc's rows");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int part = wave / WPD, d = (wave % WPD) * 64 + lane;
  const float *ml = p.ws_ml + (bh * p.splits + min(lane, p.splits - 1)) * 2;
  float ms = __hip_atomic_load(ml, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const float ls = __hip_atomic_load(ml + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const float *orow = p.ws_o + bh * p.splits * D + d;
  float o = 0.0f, wgt = 0.0f, lt = 0.0f;
  for (int s0 = part; s0 < p.splits; s0 += R * PARTS) {  // wave-uniform
    float os[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
      os[r] = __hip_atomic_load(orow + (int64_t)min(s0 + r * PARTS, p.splits - 1) * D, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
    if (s0 == part) {  // the weights, under the loads of the first rows
      if (lane >= p.splits) ms = -INFINITY;
      const float mx = wave_max(ms);
      wgt = ms == -INFINITY ? 0.0f : fast_exp2(ms - mx);
      lt = lane < p.splits ? ls * wgt : 0.0f;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) lt += shfl_xor(lt, off);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int s = s0 + r * PARTS;
      const float f = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(wgt), min(s, 63)));
      o += s < p.splits ? os[r] * f : 0.0f;
    }
  }
  s_acc[part][d] = o;  // every thread read s_acc before the barriers above
  __syncthreads();
  if (part != 0) return;
#pragma unroll
  for (int k = 1; k < PARTS; ++k) o += s_acc[k][d];
  p.out[bh * D + d] = (half_t)(lt > 0.0f ? o / lt : 0.0f);
}

// Split count used by the decode kernels for this launch shape.
int decode_splits(int32_t batch, int32_t heads, int32_t max_pages_visited, bool int4);
// Launches the split-K INT4 decode kernel (splits merged in-kernel); `pages`:
// the pages a sequence may visit.
int launch_decode_int4(const DecodeParams &p, int32_t batch, int32_t D, int32_t scale_dtype, int32_t pages,
                       hipStream_t stream);

// Launches the split-K fp16-pool decode kernel (splits merged in-kernel).
int launch_decode_fp16(const DecodeParams &p, int32_t batch, int32_t D, hipStream_t stream);

// Multi-query (q_len >= 2) MFMA kernel over INT4 page pools or contiguous
// fp16 pools with 16-multiple pages and D in {64, 128}.
bool prefill_supported(const memopt_attn_desc &d);
// Workspace of the staged prefill path (0: the path stages in-kernel).
int64_t prefill_workspace_bytes(const memopt_attn_desc &d);
int64_t staged_copy_bytes(const memopt_attn_desc &d);  // the same, also past the sizes the staged path takes
int launch_prefill(const memopt_attn_desc &d, int32_t W, float qk_scale_log2, hipStream_t stream);

// Multi-query kernel without staging (direct.hip): calls over INT4 pages and
// fp16 pools that it is estimated to run faster than the staged path, and any
// number of queries over token-major INT4 codes (D in {64, 128}, pages of a
// multiple of 16 tokens, aligned strides).
bool direct_supported(const memopt_attn_desc &d);
// Bytes of split-K partials; a call that has less room runs fewer splits.
int64_t direct_workspace_bytes(const memopt_attn_desc &d);
int launch_direct(const memopt_attn_desc &d, int32_t W, float qk_scale_log2, hipStream_t stream);

// CUs of the current device (looked up once).
int compute_units();

}  // namespace memopt
