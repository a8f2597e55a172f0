// Single-token decode attention with per-key score-sums for gfx950 (HBM-bound).
//
// Reference behaviour: keys_values/attention/flashinfer_ops.py:193-275 (sdpa_decode: no mask, the
// weights divided by the group size), keys_values/csrc/kernels/sdpa_decode.cu:616-898 (the kernel
// it calls, which reads K and V once per QUERY head and keeps fp32 logits to turn them into
// weights afterwards, :838-854).
//
// Here one workgroup serves all G query heads of a (batch, KV head, split), so K and V cross HBM
// once, in one pass with both streams in flight: 8 or 16 lanes share a row (a lane owns 8 consecutive
// d, 16-byte loads, a wavefront instruction covers whole contiguous rows of K or V), the G logits of
// a row are v_dot2_f32_bf16 sums reduced over the row's lanes with DPP adds, and O += p V runs on
// the same lanes with dot2 over pairs of rows. Every row group of a wavefront keeps its own running
// maximum, sum and fp32 accumulator (the maximum moves lazily), so the loop has no barrier and no
// cross-lane traffic beyond the row reduction; groups and wavefronts are merged once at the end.
// The logits (log2 units) of a split are gathered in LDS, [key][head]. When a split's logits fit there
// (16384 / G keys for most shapes), they never leave the chip: a workgroup publishes its partial maximum and sum, polls
// until the other splits of its (batch, KV head) row have done the same (workgroups are dispatched in
// index order and a row's splits are neighbours, so they run at the same time; the wait is bounded),
// combines them into the row's base-2 log-sum-exp and turns its own logits into
// W = (1/G) sum_g exp2(logit_g - lse_g) on the spot; in the fused H2O form it also adds W to the cumulative
// scores and feeds the row's lowest-score slot. Longer splits, and a workgroup whose wait ran out, send the
// logits to an fp32 scratch in bursts of 32 KB (a write stream mixed into the reads costs HBM far more than
// its share of the bytes). The splits of a row also combine its outputs, each an equal share, and the one that
// finishes last publishes the chosen slot (finish_split). Only where the logits go through the scratch by plan one more
// launch follows: some of its workgroups combine the splits' outputs, the others do the weights work, and the one that
// finishes last publishes the chosen slots. K and V are touched once: they are loaded non-temporally. No float
// atomics anywhere.
// Quantised stores, and plain rows with 8 to 16 query heads per KV head, take a second form of the split kernel
// (decode_mfma_kernel, below) that does both products on the matrix cores: with codes to dequantise, or with that
// many dot products per loaded value, the form above is bound by its vector arithmetic, not by HBM.
// The kernels and their launch; sdpa_decode.hip plans the calls, one sdpa_decode_<D>.hip per head size instantiates launch_d.
#pragma once
#include <type_traits>

#include "key_blocks.h"

namespace kvx {
namespace decode {

constexpr int NTHREADS = 256;
constexpr int WAVES = 4;

struct DecodeParams {
  const uint16_t* q;
  const void* k;
  const void* v;
  const float* k_scale;
  const int32_t* k_zp;
  const float* v_scale;
  const int32_t* v_zp;
  uint16_t* o;
  float* lse_out;  // user (B, 1, Hq) or NULL
  float* w;        // user (B, Hkv, kv_len) or NULL
  float* logits;   // (B, Hkv, Tpad, G), G the padded group size
  float* part_o;   // (B, Hkv, S, Gr, D)
  float* part_ml;  // (B, Hq, S, 2): maximum and sum of a split; one-launch form: zero until the split has published them
  // one-launch form (everything but logits that go through the scratch by plan):
  uint32_t* row_count;            // a line per (b, kvh) row: [kArrived] splits whose outputs (part_o) are there,
                                  // [kFinished] splits whose choice and split_pending are there (their reads of part_o may be on the way)
  unsigned long long* part_best;  // (B, Hkv, S): (value, slot) minimum of the split's keys (fused H2O form)
  float* part_vn;                 // (B, Hq, S): sum of |V row| 2^(logit - maximum) (scores weighted by the V norms)
  float* part_stats;              // (B, Hkv, S, 4): extremes of the compared value and of the quantisation errors
  uint32_t* split_pending;        // (B, Hkv, S): what a split whose wait ran out left to the row's last one (finish_split)
  // logits through the scratch by plan, two launches:
  unsigned long long* best;  // fused H2O form: (value, slot) minimum per (b, kvh) row, else NULL
  uint32_t* tail_count;      // fused H2O form: workgroups of the tail kernel's second kind that have finished
  uint32_t* scratch_splits;  // caller's counter of the splits whose logits went through the scratch, or NULL
  int32_t qs_vec;            // quantiser state arrays are 16-byte aligned with strides that keep them so (vector loads of 4 keys)
  int32_t resident;          // the logits of a split stay in LDS
  int32_t one_launch;        // the splits themselves combine their outputs (always, but for logits through the scratch by plan)
  int32_t spin_limit;        // polls of the other splits' pairs before a workgroup gives up and sends its logits out
  int32_t poll_sleep;        // pause between two polls, in units of 512 cycles
  int32_t B, Hq, Hkv, kv_len, Tpad, num_splits, keys_per_split;
  int32_t Gr;  // query heads per KV head; the kernels' G is Gr rounded up to a power of two (heads Gr .. G - 1 are
               // dummies: zero queries, nothing of theirs is stored, their logits count for nothing)
  int32_t share;  // value pairs of a row's outputs that a split combines: ceil(Gr D / 2 / num_splits)
  int32_t scores, positions;  // fused H2O form: scores are kept; compared per token position
  int32_t lj;     // log2 of the lanes that share a pair there
  float c, inv_g;  // inv_g = 1 / Gr
  int64_t q_sb, q_sh, k_sb, k_sh, k_st, v_sb, v_sh, v_st, o_sb, o_sh, qs_sb, qs_sh;
};


// Sum over the LPR lanes that share a row. Every lane of the group ends with the same bits: each
// step adds two values that the partner lane adds in the other order.
template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
  return x + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, false));
}
template <int LPR>
__device__ __forceinline__ float row_group_sum(float x) {
  static_assert(LPR == 32 || LPR == 16 || LPR == 8, "row groups of 8, 16 or 32 lanes");
  if constexpr (LPR == 32) x += __shfl_xor(x, 16, 64);  // the other DPP row of the group
  if constexpr (LPR >= 16) {
    x = dpp_add<0x128>(x);  // row_ror:8
    x = dpp_add<0x124>(x);  // row_ror:4
  } else {
    x = dpp_add<0x141>(x);  // row_half_mirror
  }
  x = dpp_add<0x4E>(x);  // quad_perm [2,3,0,1]
  x = dpp_add<0xB1>(x);  // quad_perm [1,0,3,2]
  return x;
}

// Exchanges between the 16-lane rows and the halves of a wavefront on the vector ALU (v_permlane16_swap,
// v_permlane32_swap: the odd rows (the upper half) of the first operand change places with the even rows (the lower
// half) of the second).
__device__ __forceinline__ float dpp_ror8(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x128, 0xf, 0xf, false));
}
// even rows: sum of a over the row pair, odd rows: sum of b over it
__device__ __forceinline__ float swap_rows_add(float a, float b) {
  const u32pair_t r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float sum_row_pairs(float v) { return swap_rows_add(v, v); }
// lower half: sum of a over the two halves, upper half: sum of b
__device__ __forceinline__ float swap_halves_add(float a, float b) {
  const u32pair_t r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Over the whole wavefront, every lane with the same bits (each step joins two values that the partner joins in the other
// order), on the vector ALU: behind the key loop a step of such a reduction is waited for, and six through LDS take 0.3 us.
__device__ __forceinline__ float wave_sum(float x) {
  x = dpp_add<0x128>(x);  // row_ror:8
  x = dpp_add<0x124>(x);  // row_ror:4
  x = dpp_add<0x4E>(x);   // quad_perm [2,3,0,1]
  x = dpp_add<0xB1>(x);   // quad_perm [1,0,3,2]
  return sum_halves(sum_row_pairs(x));
}
template <int CTRL>
__device__ __forceinline__ float dpp_max(float x) {
  return fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, false)));
}
__device__ __forceinline__ float wave_max(float x) {
  x = dpp_max<0xB1>(dpp_max<0x4E>(dpp_max<0x124>(dpp_max<0x128>(x))));
  return max_halves(max_row_pairs(x));
}
__device__ __forceinline__ float wave_min(float x) { return -wave_max(-x); }
__device__ __forceinline__ unsigned long long join_words(uint32_t lo, uint32_t hi) { return ((unsigned long long)hi << 32) | lo; }
template <int CTRL>
__device__ __forceinline__ unsigned long long dpp_min(unsigned long long x) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)x, CTRL, 0xf, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(x >> 32), CTRL, 0xf, 0xf, false);
  return min(x, join_words(lo, hi));
}
__device__ __forceinline__ unsigned long long wave_min(unsigned long long x) {
  x = dpp_min<0xB1>(dpp_min<0x4E>(dpp_min<0x124>(dpp_min<0x128>(x))));
  u32pair_t lo = __builtin_amdgcn_permlane16_swap((uint32_t)x, (uint32_t)x, false, false);
  u32pair_t hi = __builtin_amdgcn_permlane16_swap((uint32_t)(x >> 32), (uint32_t)(x >> 32), false, false);
  x = min(join_words(lo[0], hi[0]), join_words(lo[1], hi[1]));
  lo = __builtin_amdgcn_permlane32_swap((uint32_t)x, (uint32_t)x, false, false);
  hi = __builtin_amdgcn_permlane32_swap((uint32_t)(x >> 32), (uint32_t)(x >> 32), false, false);
  return min(join_words(lo[0], hi[0]), join_words(lo[1], hi[1]));
}

// Logits a workgroup holds in LDS, in whole pairs of steps of the widest kernel (256 keys). Two workgroups per compute
// unit share 160 KB of LDS: the logits take what the merge buffer (4 G D floats) leaves of 80 KB. At head size 256 the
// kernel over codes takes 320 to 370 registers and has its compute unit to itself: the logits take what is left of the
// whole 160 KB, so that rows of many heads run in one round of splits instead of three (16 rows of 35407 8-bit keys, 7 heads
// each, with weights: 133 -> 73 us).
constexpr int logit_floats(int G, int D, bool codes) {
  if (D == 256 && codes) return G == 8 ? 30720 : 32768;
  return G * D <= 512 ? 16384 : (G * D <= 1024 ? (G == 16 ? 12288 : 14336) : 8192);
}
constexpr int kMaxSplits = 512;  // of a row
// The weights of a row's splits (finish_split) take the LDS of the wavefronts' outputs, which has room for WAVES * D of them a head:
// for all at head sizes from 128 on, for 256 at 64. Those of more splits take the place of the logits, once these are used; a
// buffer of their own would leave a compute unit one workgroup of 16 heads instead of two.
constexpr bool weights_beside_logits(int D, int S) { return WAVES * D >= kMaxSplits || S <= WAVES * D; }
constexpr int kCountStride = 64;  // a row's counters have 256 bytes to themselves: the polls of different rows go to different channels
constexpr int kArrived = 0, kFinished = 1, kSelected = 2;
static_assert(kCountStride == kDecodeCounterStride, "the slot write clears these counters");
constexpr uint32_t kPending = 1u << 16;  // added to kFinished by a split that leaves its weights to the row's last one
constexpr float kNegBig = -1.0e30f;  // running maximum before the first key (finite: no inf - inf)
constexpr float kRescaleSlack = 8.0f;  // the running maximum moves only when a logit exceeds it by this

// Monotone map float -> uint32 (a < b  <=>  key(a) < key(b)); -0.0 is folded onto +0.0.
__device__ __forceinline__ uint32_t ordered_bits(float x) {
  x += 0.0f;
  const uint32_t u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Maximum and sum (relative to it) of a query head from its splits' (maximum, sum) pairs, by one wavefront: lane s adds
// splits s, s + 64, ..., then the lanes are joined; every lane ends with the same bits. The outputs are scaled by these two:
// the log-sum-exp, one number, is rounded at the size of the logits (at 10^6 by 2^-5, 2 % of a weight).
struct RowSum {
  float top = -INFINITY, sum = 0.0f;
  __device__ __forceinline__ void add(unsigned long long pair) {
    const float m = __uint_as_float((uint32_t)pair), l = __uint_as_float((uint32_t)(pair >> 32));
    const float mn = fmaxf(top, m);
    if (mn > -INFINITY) sum = sum * fast_exp2(top - mn) + l * fast_exp2(m - mn);
    top = mn;
  }
  __device__ __forceinline__ void join_lanes() {
    const float mw = wave_max(top);
    sum = wave_sum(top > -INFINITY ? sum * fast_exp2(top - mw) : 0.0f);
    top = mw;
  }
  __device__ __forceinline__ float lse() const { return top + fast_log2(sum); }  // base 2
};
constexpr unsigned long long kEmptyPair = 0xff800000ull;  // (maximum -inf, sum 0)
// of a head whose pairs an earlier launch left
__device__ __forceinline__ RowSum row_sum(const float* part_ml, int num_splits, int lane) {
  RowSum r;
  for (int sp = lane; sp < num_splits; sp += 64) r.add(((const unsigned long long*)part_ml)[sp]);
  r.join_lanes();
  return r;
}

// The logits gathered in LDS leave as one contiguous burst (keys past the end of a chunk of CHUNK keys are -inf).
template <int G, int LGK, int CHUNK>
__device__ __forceinline__ void flush_logits(const float* lgbuf, float* lgrow, int lg_base, int k_end, int tid) {
  const int nkeys = min(LGK, (k_end - lg_base + CHUNK - 1) / CHUNK * CHUNK);
  f32x4_t* dst = (f32x4_t*)(lgrow + (int64_t)lg_base * G);
  for (int j = tid; j < nkeys * G / 4; j += NTHREADS) dst[j] = ((const f32x4_t*)lgbuf)[j];
}

// Values that cross workgroups inside one launch: device-coherent (they bypass the caches that the dies do not share).
template <typename P>
__device__ __forceinline__ auto coherent_load(P p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename P, typename T>
__device__ __forceinline__ void coherent_store(P p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ unsigned long long pair_bits(float lo, float hi) {
  return ((unsigned long long)__float_as_uint(hi) << 32) | __float_as_uint(lo);
}

// LDS of the part of a workgroup's life after its key loop.
template <int G>
struct FinishShared {
  float lse[G];
  float inv[G];  // 1 / sum of the head relative to its maximum
  float top[G];  // its maximum, where the splits' weights come later
  float z;  // scores weighted by the V norms: the row's sum of |V row| W
  float vn[G];
  float red[WAVES][4];
  unsigned long long best[WAVES];
  uint32_t ready[WAVES], outputs, finished;
};

// Where a workgroup's (batch, KV head) row keeps what the part behind the key loop uses. Formed before the key loop, while its
// first loads are waited for, and pinned to registers: formed where they are used, by 64-bit scalar products of strides, and with
// the flags read from the argument block as the branches come, they were a third of the instructions there (14.6 -> 12.7 us
// for the step over 8 rows of 4096 keys, with kernels of their own for the variants).
template <typename T>
using global_ptr = T __attribute__((address_space(1)))*;  // stays a global access behind the pin
struct RowAt {
  global_ptr<unsigned long long> ml;  // pairs of the row, [head][split]
  global_ptr<unsigned long long> po;  // outputs of the row in pairs, [split][Gr D / 2]
  global_ptr<uint32_t> cnt, pending;  // counters of the row, what its splits left
  global_ptr<unsigned long long> best;  // choices of the row's splits
  global_ptr<float> w, sc;            // weights and scores of the row, where there are any
  global_ptr<int32_t> pos;            // token positions, where scores are compared per position
  global_ptr<uint16_t> o;             // outputs of the row's first head
};
template <typename T>
__device__ __forceinline__ void set_pinned(global_ptr<T>& to, T* x) {
  to = (global_ptr<T>)x;
  asm volatile("" : "+v"(to));  // vector registers: the scalar ones are short
}
template <int D>
__device__ __forceinline__ RowAt row_at(const DecodeParams& p, const kvx_h2o_args& hh, const int b, const int kvh) {
  const int row = b * p.Hkv + kvh, S = p.num_splits;
  RowAt at;
  set_pinned(at.ml, (unsigned long long*)p.part_ml + (int64_t)row * (p.Gr * S));
  set_pinned(at.po, (unsigned long long*)p.part_o + (int64_t)row * (S * p.Gr) * (D / 2));
  set_pinned(at.cnt, p.row_count + row * kCountStride);
  set_pinned(at.pending, p.split_pending + (int64_t)row * S);
  set_pinned(at.best, p.part_best + (int64_t)row * S);
  set_pinned(at.w, p.w + (int64_t)row * p.kv_len);
  set_pinned(at.sc, hh.scores + (b * hh.sc_stride_b + kvh * hh.sc_stride_h));
  set_pinned(at.pos, (int32_t*)hh.token_pos + (b * hh.tp_stride_b + kvh * hh.tp_stride_h));
  set_pinned(at.o, p.o + (b * p.o_sb + (int64_t)(kvh * p.Gr) * p.o_sh));
  return at;
}
template <typename P>
__device__ __forceinline__ P at_byte(P base, uint32_t bytes) {
  return (P)((global_ptr<char>)base + bytes);
}

// Maximum of a head in a split, by its place in [head][split], once the pairs have been found.
__device__ __forceinline__ float split_maximum(const RowAt& at, const int i) { return __uint_as_float((uint32_t)coherent_load(at_byte(at.ml, (uint32_t)i * 8u))); }

// The row's maxima, sums and log-sum-exps (and z) from its splits' partials, in LDS for the whole workgroup, and every split's
// weight 2^(maximum - row's maximum) in wt ([head][split]; unless early, late_weights forms these). wait: the splits may still be
// on their way. The pairs themselves say so: they are zero before the launch and never afterwards, so a poll that finds them all has them already (a count of the
// splits that have arrived costs a wait for the pairs' store, the atomic add behind it and, once the count is full, another
// read: 1 us of a 16 us step). Bounded; returns whether all were found.
template <int G, bool VARIANT>
__device__ __forceinline__ bool row_state(const DecodeParams& p, const RowAt& at, const bool wait, const bool vnorm, const int row, FinishShared<G>& sh, float* wt,
                                          const bool early) {
  constexpr int HPW = (G + WAVES - 1) / WAVES;  // heads of a wavefront: wave, wave + WAVES, ...; lane s takes splits s, s + 64, ...
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), S = p.num_splits;
  RowSum rs[HPW];
  bool ok = p.spin_limit > 0 || !wait;
  int spin = 0;
  for (int base = 0; base < S && ok; base += 64) {
    const int sp = base + lane;
    unsigned long long pair[HPW];
    for (;;) {
      bool all = true;
#pragma unroll
      for (int h = 0; h < HPW; ++h) {
        const int g = wave + WAVES * h;
        pair[h] = kEmptyPair;
        if (g < p.Gr && sp < S) pair[h] = coherent_load(at_byte(at.ml, (uint32_t)(g * S + sp) * 8u));
      }
#pragma unroll
      for (int h = 0; h < HPW; ++h) all = all && pair[h] != 0;
      if (__all(all) || !wait) break;
      if (++spin >= p.spin_limit) {
        ok = false;
        break;
      }
      // short pauses first: splits of a row that run side by side arrive within a microsecond of each other
      const int pause = min(p.poll_sleep, 1 + (spin >> 2));
      for (int z = 0; z < pause; ++z) __builtin_amdgcn_s_sleep(8);
    }
#pragma unroll
    for (int h = 0; h < HPW; ++h) {
      const int g = wave + WAVES * h;
      rs[h].add(pair[h]);
      if (early && g < G && sp < S) wt[g * S + sp] = __uint_as_float((uint32_t)pair[h]);
    }
  }
#pragma unroll
  for (int h = 0; h < HPW; ++h) {
    const int g = wave + WAVES * h;
    if (g >= G) break;
    rs[h].join_lanes();
    const float lse = g < p.Gr ? rs[h].lse() : INFINITY;  // dummy heads: exp2(x - inf) = 0
    float z = 0.0f;
    if (__builtin_expect(early, 1)) {
      for (int sp = lane; sp < S; sp += 64) {  // the lane's own entries
        const float m = wt[g * S + sp];
        if constexpr (VARIANT)
          if (vnorm && g < p.Gr && ok) z += coherent_load(p.part_vn + ((int64_t)row * p.Gr + g) * S + sp) * fast_exp2(m - lse);
        wt[g * S + sp] = fast_exp2(m - rs[h].top);
      }
    } else {
      if constexpr (VARIANT)
        if (vnorm && g < p.Gr && ok)
          for (int sp = lane; sp < S; sp += 64) z += coherent_load(p.part_vn + ((int64_t)row * p.Gr + g) * S + sp) * fast_exp2(split_maximum(at, g * S + sp) - lse);
      if (lane == 0) sh.top[g] = rs[h].top;
    }
    if (VARIANT && vnorm) z = wave_sum(z);
    if (lane == 0) {
      sh.lse[g] = lse;
      sh.inv[g] = 1.0f / rs[h].sum;
      if (VARIANT) sh.vn[g] = z;
    }
  }
  if (lane == 0) sh.ready[wave] = ok;
  __syncthreads();
  static_assert(WAVES == 4, "the wavefronts' answers");
  ok = sh.ready[0] && sh.ready[1] && sh.ready[2] && sh.ready[3];
  if (VARIANT && vnorm) {
    if (threadIdx.x == 0) {
      float z = 0.0f;
      for (int g = 0; g < p.Gr; ++g) z += sh.vn[g];
      sh.z = z / (float)p.Gr;
    }
    __syncthreads();
  }
  return ok;
}

// The splits' weights behind row_state, for the whole workgroup.
template <int G>
__device__ __forceinline__ void late_weights(const DecodeParams& p, const RowAt& at, const FinishShared<G>& sh, float* wt) {
  for (int g = 0; g < p.Gr; ++g)
    for (int sp = threadIdx.x; sp < p.num_splits; sp += NTHREADS) wt[g * p.num_splits + sp] = fast_exp2(split_maximum(at, g * p.num_splits + sp) - sh.top[g]);
  __syncthreads();
}

// The row's outputs for the value pairs [e0, e1) of its E = Gr D / 2: O = (sum over the splits of part_o weight) / sum. J
// neighbouring lanes share a pair, lane j taking splits j, j + J, ... (at most four loads a lane up to 64 splits: one memory
// latency a pass); their sums are added in a fixed order, so the result does not depend on which workgroup takes
// which pairs. `asked` runs once, when the loads of the first pass are on their way.
template <int D, bool F16, int G, typename FN>
__device__ __forceinline__ void merge_pairs(const DecodeParams& p, const RowAt& at, const FinishShared<G>& sh, const float* wt, const int e0, const int e1, FN asked) {
  const int tid = threadIdx.x, S = p.num_splits, lj = p.lj, J = 1 << lj, j = tid & (J - 1);
  const uint32_t step = (uint32_t)(p.Gr * (D / 2)) * 8u;  // byte offsets fit 32 bits: at most 512 splits x 16 heads x 256 floats
  bool first = true;
  for (int base = e0; base < e1 || first; base += NTHREADS >> lj) {
    const int e = base + (tid >> lj);
    const bool live = e < e1;
    unsigned long long x[4];
    auto load = [&](int s0) {
#pragma unroll
      for (int u = 0; u < 4; ++u) x[u] = coherent_load(at_byte(at.po, (uint32_t)min(s0 + J * u, S - 1) * step + (uint32_t)e * 8u));
    };
    if (live) load(j);
    if (first) asked();
    first = false;
    f32x2_t acc = {0.0f, 0.0f};
    const int g = live ? e / (D / 2) : 0;
    if (live)
      for (int s0 = j; s0 < S; s0 += 4 * J) {
        if (s0 != j) load(s0);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float w = s0 + J * u < S ? wt[g * S + s0 + J * u] : 0.0f;
          acc[0] += __uint_as_float((uint32_t)x[u]) * w;
          acc[1] += __uint_as_float((uint32_t)(x[u] >> 32)) * w;
        }
      }
    auto join = [&](auto ctrl) {
      acc[0] = dpp_add<decltype(ctrl)::value>(acc[0]);
      acc[1] = dpp_add<decltype(ctrl)::value>(acc[1]);
    };
    if (lj >= 1) join(std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
    if (lj >= 2) join(std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
    if (lj >= 3) join(std::integral_constant<int, 0x141>{});  // row_half_mirror
    if (lj >= 4) join(std::integral_constant<int, 0x140>{});  // row_mirror
    if (j == 0 && live) {
      const float inv = sh.inv[g];
      *(global_ptr<uint32_t>)(at.o + (int64_t)g * p.o_sh + 2 * (e % (D / 2))) = pack_pair<F16>(acc[0] * inv, acc[1] * inv);
    }
  }
}

// What the cache keeps of four keys of a thread (k, k + NTHREADS, ...): the scores to add to and what goes into the choice.
template <bool VARIANT>
struct KeyState {
  float score[4];
  int32_t pos[4];
  float v_norm[VARIANT ? 4 : 1], q_error[VARIANT ? 4 : 1];
  __device__ __forceinline__ void load(const RowAt& at, const bool positions, const float* vn, const float* qe, const int k, const int k_end) {
    uint32_t ku[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) ku[u] = (uint32_t)min(k + u * NTHREADS, k_end - 1) * 4u;
#pragma unroll
    for (int u = 0; u < 4; ++u) score[u] = *at_byte(at.sc, ku[u]);
    if (positions) {
#pragma unroll
      for (int u = 0; u < 4; ++u) pos[u] = *at_byte(at.pos, ku[u]);
    }
    if constexpr (VARIANT) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        v_norm[u] = vn ? *at_byte((global_ptr<const float>)vn, ku[u]) : 0.0f;
        q_error[u] = qe ? *at_byte((global_ptr<const float>)qe, ku[u]) : 0.0f;
      }
    }
  }
};
// Of the keys a thread has weighed: their (value, slot) minimum, or, where the compared value is normalised over the batch
// element before the choice, its extremes and those of the errors.
template <bool VARIANT>
struct Choice {
  unsigned long long best = ~0ull;
  float smin = INFINITY, smax = -INFINITY, qmin = INFINITY, qmax = -INFINITY;
};

// One key of a thread: W from its logits x, and in the fused H2O form scores += W (or the V-norm weighted increment).
template <int G, bool VARIANT>
__device__ __forceinline__ void weigh_key(const DecodeParams& p, const kvx_h2o_args& hh, const RowAt& at, const float (&lse)[G], const float z, const int k, const float* x,
                                          const KeyState<VARIANT>& ks, const int u, Choice<VARIANT>& c) {
  float acc = 0.0f;
#pragma unroll
  for (int g = 0; g < G; ++g) acc += fast_exp2(x[g] - lse[g]);
  acc *= p.inv_g;
  if (p.w) *at_byte(at.w, (uint32_t)k * 4u) = acc;
  if (!p.scores) return;
  // every product and sum rounded on its own, as the reference's tensor expressions are
  float inst = acc;
  if constexpr (VARIANT)
    if (hh.v_norm) inst = __fmul_rn(__fmul_rn(ks.v_norm[u], acc) / z, (float)hh.q_len);
  float val = __fadd_rn(ks.score[u], inst);
  *at_byte(at.sc, (uint32_t)k * 4u) = val;
  if (k >= hh.limit) return;
  if (p.positions) val = val / (float)(hh.input_pos - max(ks.pos[u], hh.prefill_len - 1));
  if constexpr (VARIANT)
    if (hh.q_errors) {
      c.smin = fminf(c.smin, val);
      c.smax = fmaxf(c.smax, val);
      c.qmin = fminf(c.qmin, ks.q_error[u]);
      c.qmax = fmaxf(c.qmax, ks.q_error[u]);
      return;
    }
  c.best = min(c.best, join_words((uint32_t)k, ordered_bits(val)));
}
// per wavefront in sh, for publish_choice behind a barrier
template <int G, bool VARIANT>
__device__ __forceinline__ void leave_choice(const kvx_h2o_args& hh, FinishShared<G>& sh, Choice<VARIANT>& c) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if constexpr (VARIANT)
    if (hh.q_errors) {
      const float r[4] = {wave_min(c.smin), wave_max(c.smax), wave_min(c.qmin), wave_max(c.qmax)};
      if (lane == 0)
        for (int i = 0; i < 4; ++i) sh.red[wave][i] = r[i];
      return;
    }
  c.best = wave_min(c.best);
  if (lane == 0) sh.best[wave] = c.best;
}
template <int G, bool VARIANT>
__device__ __forceinline__ void publish_choice(const DecodeParams& p, const kvx_h2o_args& hh, const RowAt& at, FinishShared<G>& sh, const int row, const int split) {
  const int tid = threadIdx.x;
  if constexpr (VARIANT)
    if (hh.q_errors) {
      if (tid < 4) {
        float r = sh.red[0][tid];
        for (int i = 1; i < WAVES; ++i) r = (tid & 1) ? fmaxf(r, sh.red[i][tid]) : fminf(r, sh.red[i][tid]);
        p.part_stats[((int64_t)row * p.num_splits + split) * 4 + tid] = r;  // read by the next launch
      }
      return;
    }
  if (tid == 0) {
    unsigned long long mn = sh.best[0];
#pragma unroll
    for (int i = 1; i < WAVES; ++i) mn = min(mn, sh.best[i]);
    coherent_store(at_byte(at.best, (uint32_t)split * 8u), mn);
  }
}

// What a split does once its wavefronts have left their partial results in LDS (red: unnormalised outputs, rml:
// maximum and sum, per wavefront and head).
//
// One launch does the whole step. The split publishes its partial and waits (boundedly) for the maxima and sums of the row's
// others; with weights wanted it turns its own logits (lgbuf, [key][head]) into weights while the others' outputs arrive, then
// takes an equal share of the row's outputs. A split whose wait ran out puts its logits into the scratch instead. The split that
// finishes last makes up what such splits left undone and publishes the row's slot. A second launch for the outputs and a third
// to reset the counters cost 4 to 8 us of every step, a third of a step over 4096 slots.
// What bounds this part is latency: waits for memory that the dies share, 0.4 to 0.6 us each, and the instructions between them,
// which a wavefront that has its SIMD to itself issues one in five cycles or so. So what can be asked for early is (the
// scores before the wait, the outputs' count before the weights), a store that others wait for is followed by other work, and
// the policies that weigh scores in other ways have kernels of their own (VARIANT). Whole steps, with a count of arrivals waited
// for by one lane, one key weighed a pass and reductions through LDS -> as here: 8 rows of 4096 keys 16.2 -> 12.7 us, 32 rows
// of 16384 8-bit keys 44.0 -> 40.9.
template <int D, int G, bool F16, bool VARIANT>
__device__ __forceinline__ void finish_split(const DecodeParams& p, const kvx_h2o_args& hh, const RowAt& at, float* lgbuf, float (&red)[WAVES][G][D],
                                             const float (&rml)[WAVES][G][2], float* lgrow, const int k_begin, const int k_end) {
  __shared__ FinishShared<G> sh;
  static_assert(WAVES * D >= kMaxSplits || G * kMaxSplits <= logit_floats(G, D, true), "late weights take the logits' place");
  const int tid = threadIdx.x;
  const int split = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
  const int row = b * p.Hkv + kvh, S = p.num_splits, E = p.Gr * (D / 2);
  const bool vnorm = VARIANT && hh.v_norm;
  const float* vn = vnorm ? hh.v_norm + b * hh.sc_stride_b + kvh * hh.sc_stride_h : nullptr;
  const float* qe = VARIANT && hh.q_errors ? hh.q_errors + b * hh.sc_stride_b + kvh * hh.sc_stride_h : nullptr;
  const bool early = weights_beside_logits(D, S);
  float* wt = early ? &red[0][0][0] : lgbuf;  // [head][split]
  auto publish_sums = [&] {   // read by other workgroups while this kernel runs, as are the outputs
    if (tid < p.Gr) {
      float M = rml[0][tid][0], l = 0.0f;
#pragma unroll
      for (int w = 1; w < WAVES; ++w) M = fmaxf(M, rml[w][tid][0]);
#pragma unroll
      for (int w = 0; w < WAVES; ++w) l += rml[w][tid][1] * fast_exp2(rml[w][tid][0] - M);
      unsigned long long pair = pair_bits(M, l);
      if (pair == 0) pair = 1;  // zero is what others wait for to change (a split's sum is at least 2^-8, or NaN)
      coherent_store(at_byte(at.ml, (uint32_t)(tid * S + split) * 8u), pair);
    }
  };
  __syncthreads();
  if (!vnorm) publish_sums();
  KeyState<VARIANT> ks;
  if (p.scores && p.one_launch) ks.load(at, p.positions, vn, qe, k_begin + tid, k_end);
  for (int i = tid; i < E; i += NTHREADS) {
    const int g = i / (D / 2), d = 2 * (i % (D / 2));
    float M = rml[0][g][0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) M = fmaxf(M, rml[w][g][0]);
    float x0 = 0.0f, x1 = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float sc = fast_exp2(rml[w][g][0] - M);
      x0 += red[w][g][d] * sc;
      x1 += red[w][g][d + 1] * sc;
    }
    coherent_store(at_byte(at.po, (uint32_t)(split * E + i) * 8u), pair_bits(x0, x1));
  }
  if (vnorm) {  // this split's part of z: sum over its keys of |V row| 2^(logit - maximum), per head; there before the sums are
    float M[G], a[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      M[g] = rml[0][g][0];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) M[g] = fmaxf(M[g], rml[w][g][0]);
      a[g] = 0.0f;
    }
    for (int k = k_begin + tid; k < k_end; k += NTHREADS) {
      const float v = vn[k];
#pragma unroll
      for (int g = 0; g < G; ++g) a[g] += v * fast_exp2(lgbuf[(k - k_begin) * G + g] - M[g]);
    }
    __syncthreads();  // red has been read
    float* part = &red[0][0][0];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      a[g] = wave_sum(a[g]);
      if ((tid & 63) == 0) part[(tid >> 6) * G + g] = a[g];
    }
    __syncthreads();
    if (tid < p.Gr) {
      float t = part[tid];
      for (int w = 1; w < WAVES; ++w) t += part[w * G + tid];
      coherent_store(p.part_vn + ((int64_t)row * p.Gr + tid) * S + split, t);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    publish_sums();  // the same lanes: behind their part of z
  }
  if (!p.one_launch) return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the outputs above have reached device-coherent memory
  __syncthreads();
  if (tid == 0 && S > 1) __hip_atomic_fetch_add(at.cnt + kArrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  bool ready = p.spin_limit > 0;
  if (S > 1 || ready) ready = row_state<G, VARIANT>(p, at, S > 1, vnorm, row, sh, wt, early);
  uint32_t left = 0, finished = 0;  // left to the row's last split: 1 the weights, 2 the outputs
  auto count_in = [&] {
    if (tid == 0) {
      coherent_store(at.pending + split, left);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this and the choice have reached device-coherent memory
      finished = left ? 1u + kPending : 1u;
      if (S > 1) finished += __hip_atomic_fetch_add(at.cnt + kFinished, finished, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  };
  if (ready) {
    uint32_t arrived = (uint32_t)S;
    if (tid == 0 && S > 1) arrived = coherent_load(at.cnt + kArrived);
    if (lgrow) {
      float lse[G];
#pragma unroll
      for (int g = 0; g < G; ++g) lse[g] = sh.lse[g];
      const float z = VARIANT ? sh.z : 0.0f;
      Choice<VARIANT> c;
      for (int kb = k_begin;; kb += 4 * NTHREADS) {
        const bool more = kb + 4 * NTHREADS < k_end;
        KeyState<VARIANT> next;
        if (p.scores && more) next.load(at, p.positions, vn, qe, kb + 4 * NTHREADS + tid, k_end);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int k = kb + u * NTHREADS + tid;
          if (k >= k_end) break;
          weigh_key<G, VARIANT>(p, hh, at, lse, z, k, lgbuf + (k - k_begin) * G, ks, u, c);
        }
        if (!more) break;
        ks = next;
      }
      if (p.scores) leave_choice<G, VARIANT>(hh, sh, c);
    }
    if (tid == 0) {
      for (int spin = 1; arrived < (uint32_t)S && spin < p.spin_limit; ++spin) {
        __builtin_amdgcn_s_sleep(4);
        arrived = coherent_load(at.cnt + kArrived);
      }
      sh.outputs = arrived >= (uint32_t)S;
    }
    __syncthreads();
    if (__builtin_expect(!early, 0)) late_weights<G>(p, at, sh, wt);  // behind the barrier: the logits are used
    if (p.scores) publish_choice<G, VARIANT>(p, hh, at, sh, row, split);
    const int e0 = p.share * split;
    if (!sh.outputs) left = 2;
    merge_pairs<D, F16, G>(p, at, sh, wt, e0, left ? e0 : min(e0 + p.share, E), count_in);
  } else {
    left = lgrow ? 3 : 2;
    if (lgrow) {
      const int n = (k_end - k_begin) * G;
      float* dst = lgrow + (int64_t)k_begin * G;
      for (int i = tid; i < n; i += NTHREADS) coherent_store(dst + i, lgbuf[i]);
      if (tid == 0 && p.scratch_splits) atomicAdd(p.scratch_splits, 1u);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
    count_in();
  }
  if (tid == 0) sh.finished = finished;
  __syncthreads();
  finished = sh.finished;
  if ((finished & (kPending - 1u)) != (uint32_t)S) return;

  // ---- the row's last split: what the splits that gave up left, the log-sum-exps, the chosen slot -------------------
  if (finished >= kPending) {
    if (!ready) {
      row_state<G, VARIANT>(p, at, false, vnorm, row, sh, wt, early);
      if (!early) late_weights<G>(p, at, sh, wt);
    }
    for (int sp = 0; sp < S; ++sp) {
      const uint32_t todo = coherent_load(at.pending + sp);  // the same for every thread
      if (todo & 2) merge_pairs<D, F16, G>(p, at, sh, wt, p.share * sp, min(p.share * (sp + 1), E), [] {});
      if (!(todo & 1)) continue;
      const int k0 = sp * p.keys_per_split, k1 = min(k0 + p.keys_per_split, p.kv_len);
      float lse[G];
#pragma unroll
      for (int g = 0; g < G; ++g) lse[g] = sh.lse[g];
      Choice<VARIANT> c;
      for (int k = k0 + tid; k < k1; k += NTHREADS) {
        float x[G];
#pragma unroll
        for (int g = 0; g < G; ++g) x[g] = coherent_load(lgrow + (int64_t)k * G + g);
        if (p.scores) ks.load(at, p.positions, vn, qe, k, k1);
        weigh_key<G, VARIANT>(p, hh, at, lse, VARIANT ? sh.z : 0.0f, k, x, ks, 0, c);
      }
      if (p.scores) {
        leave_choice<G, VARIANT>(hh, sh, c);
        __syncthreads();
        publish_choice<G, VARIANT>(p, hh, at, sh, row, sp);
        __syncthreads();
      }
    }
  }
  if (p.lse_out && tid < p.Gr) p.lse_out[row * p.Gr + tid] = sh.lse[tid];
  if (p.scores && !qe && tid < 64) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    unsigned long long mine = ~0ull;
    for (int sp = tid; sp < S; sp += 64) mine = min(mine, coherent_load(at_byte(at.best, (uint32_t)sp * 8u)));
    mine = wave_min(mine);
    if (tid == 0) hh.next_index[row] = (int32_t)(mine & 0xffffffffull);
  }
}

template <int D, int G, int KV, bool VARIANT>
__global__ __launch_bounds__(NTHREADS) void decode_split_kernel(const DecodeParams p, const kvx_h2o_args hh) {
  constexpr bool F16 = kv_elem_f16(KV);  // element type of q, k, v, o
  constexpr int LPR = D / 8;     // lanes per row: a lane owns 8 consecutive d
  constexpr int RPI = 64 / LPR;  // rows per load instruction of a wavefront
  constexpr int U = 4;           // load instructions per step and tensor (even: rows pair up for dot2)
  constexpr int CH = U * RPI;    // keys per wavefront and step, contiguous
  constexpr int LGK = logit_floats(G, D, false) / G;  // keys whose logits are gathered in LDS before they go out in one burst
  __shared__ __align__(16) float lgbuf[LGK * G];  // [key][head]
  __shared__ __align__(16) float red[WAVES][G][D];
  __shared__ float rml[WAVES][G][2];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int kk = lane / LPR, dc = lane % LPR;
  const int split = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
  const int k_begin = split * p.keys_per_split;
  const int k_end = min(k_begin + p.keys_per_split, p.kv_len);

  uint32_t qv[G][4];  // bf16 pairs of q[head][8 dc .. 8 dc + 8]
#pragma unroll
  for (int g = 0; g < G; ++g) {
    u32x4_t t = {0u, 0u, 0u, 0u};
    if (g < p.Gr) t = *(const u32x4_t*)(p.q + b * p.q_sb + (int64_t)(kvh * p.Gr + g) * p.q_sh + 8 * dc);
#pragma unroll
    for (int e = 0; e < 4; ++e) qv[g][e] = t[e];
  }
  // Rows are addressed as a uniform base plus a 32-bit byte offset (the host checks the range). Plain rows only:
  // quantised stores take decode_mfma_kernel.
  static_assert(kv_is_plain(KV), "plain 16-bit rows");
  const uint8_t* kbase = (const uint8_t*)p.k + (b * p.k_sb + kvh * p.k_sh) * 2;
  const uint8_t* vbase = (const uint8_t*)p.v + (b * p.v_sb + kvh * p.v_sh) * 2;
  const uint32_t k_rowb = (uint32_t)p.k_st * 2, v_rowb = (uint32_t)p.v_st * 2, lane_off = 16 * dc;
  float* lgrow = p.logits ? p.logits + ((int64_t)b * p.Hkv + kvh) * p.Tpad * G : nullptr;
  int lg_base = k_begin;  // first key of the logits gathered in LDS

  // State of this lane's row group (rows kk, kk + RPI, ... of every chunk): identical in its lanes.
  float acc[G][8], m_run[G], l_run[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m_run[g] = kNegBig;
    l_run[g] = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[g][e] = 0.0f;
  }

  struct Rows {
    u32x4_t k[U], v[U];
  };
  // Rows past the end re-read the last valid row; their logits become -inf below.
  auto issue = [&](Rows& r, int chunk0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int key = min(chunk0 + u * RPI + kk, k_end - 1);
      r.k[u] = __builtin_nontemporal_load((const u32x4_t*)(kbase + ((uint32_t)key * k_rowb + lane_off)));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int key = min(chunk0 + u * RPI + kk, k_end - 1);
      r.v[u] = __builtin_nontemporal_load((const u32x4_t*)(vbase + ((uint32_t)key * v_rowb + lane_off)));
    }
  };
  auto consume = [&](Rows& r, int chunk0) {
    // logits (log2 units) of the U rows of this lane's group, all G heads
    float s[U][G];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const u32x4_t kx = r.k[u];
      const bool valid = chunk0 + u * RPI + kk < k_end;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float a = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t kw = kx[e];  // a bit_cast applied to the vector element itself reads element 0
          a = dot2_acc<F16>(kw, qv[g][e], a);
        }
        a = row_group_sum<LPR>(a) * p.c;
        s[u][g] = valid ? a : -INFINITY;
      }
    }
    if (lgrow && dc == 0 && chunk0 < k_end) {
      typedef float fV __attribute__((ext_vector_type(G >= 4 ? 4 : G)));  // a key's G logits leave in one or two stores
      float* dst = lgbuf + (chunk0 - lg_base + kk) * G;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if constexpr (G == 1) {
          dst[u * RPI] = s[u][0];
        } else {
#pragma unroll
          for (int h = 0; h < G; h += 4) {
            fV t;
#pragma unroll
            for (int g = 0; g < (G >= 4 ? 4 : G); ++g) t[g] = s[u][h + g];
            *(fV*)(dst + u * RPI * G + h) = t;
          }
        }
      }
    }
    // running maximum: moved only when some logit of the wavefront exceeds it by the slack
    float smax[G];
    bool need = false;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float mx = s[0][g];
#pragma unroll
      for (int u = 1; u < U; ++u) mx = fmaxf(mx, s[u][g]);
      smax[g] = mx;
      need |= mx > m_run[g] + kRescaleSlack;
    }
    if (__any(need)) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float mn = fmaxf(m_run[g], smax[g]);
        const float al = fast_exp2(m_run[g] - mn);
        m_run[g] = mn;
        l_run[g] *= al;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[g][e] *= al;
      }
    }
    // O += p V, two rows per dot2
#pragma unroll
    for (int u = 0; u < U; u += 2) {
      const u32x4_t xa = r.v[u], xb = r.v[u + 1];
      uint32_t pg[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float pa = fast_exp2(s[u][g] - m_run[g]);
        const float pb = fast_exp2(s[u + 1][g] - m_run[g]);
        l_run[g] += pa + pb;
        pg[g] = pack_pair<F16>(pa, pb);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t lo = __builtin_amdgcn_perm(xb[e], xa[e], 0x05040100u);
        const uint32_t hi = __builtin_amdgcn_perm(xb[e], xa[e], 0x07060302u);
#pragma unroll
        for (int g = 0; g < G; ++g) {
          acc[g][2 * e] = dot2_acc<F16>(lo, pg[g], acc[g][2 * e]);
          acc[g][2 * e + 1] = dot2_acc<F16>(hi, pg[g], acc[g][2 * e + 1]);
        }
      }
    }
  };

  // Two steps in flight per wavefront: the loads of step i + 1 are issued before step i is consumed.
  const int nsteps = (k_end - k_begin + CH * WAVES - 1) / (CH * WAVES);
  const int stride = CH * WAVES;
  int chunk = k_begin + wave * CH;
  constexpr int FLUSH_STEPS = LGK / (CH * WAVES);
  static_assert(FLUSH_STEPS >= 2 && FLUSH_STEPS % 2 == 0, "the loop below advances two steps at a time");
  Rows ra, rb;
  issue(ra, chunk);
  const RowAt at = row_at<D>(p, hh, b, kvh);
  for (int i = 0; i + 1 < nsteps; i += 2) {
    issue(rb, chunk + stride);
    __builtin_amdgcn_sched_barrier(0);
    consume(ra, chunk);
    __builtin_amdgcn_sched_barrier(0);  // the loads below reuse the registers consumed above
    issue(ra, chunk + 2 * stride);
    __builtin_amdgcn_sched_barrier(0);
    consume(rb, chunk + stride);
    __builtin_amdgcn_sched_barrier(0);
    chunk += 2 * stride;
    if (lgrow && !p.resident && ((i + 2) % FLUSH_STEPS == 0 || i + 2 >= nsteps)) {
      __syncthreads();
      flush_logits<G, LGK, CH>(lgbuf, lgrow, lg_base, k_end, tid);
      lg_base += LGK;
      __syncthreads();
    }
  }
  // the last of an odd number of steps on its own: with the loads and the work of a second one, splits of one step took 1 us longer.
  // Out of line: an even number of steps goes on without fetching past it.
  if (__builtin_expect(nsteps & 1, 0)) {
    consume(ra, chunk);
    if (lgrow && !p.resident) {
      __syncthreads();
      flush_logits<G, LGK, CH>(lgbuf, lgrow, lg_base, k_end, tid);
    }
  }

  // ---- merge the RPI row groups of the wavefront, then the wavefronts, into one partial -----------
  // Sums over the groups by swapping register halves between lanes (reduce-scatter): at each level a lane keeps half of
  // its values, so 8 values take 8 swaps and adds instead of 16 shuffles and adds. (This code runs once per split,
  // from a cold instruction cache; with shuffles it took 3.2 us of a 15 us split of 256 keys.)
#pragma unroll
  for (int g = 0; g < G; ++g) {
    float M = m_run[g];
    if constexpr (LPR == 8) M = fmaxf(M, dpp_ror8(M));
    if constexpr (LPR <= 16) M = max_row_pairs(M);
    M = max_halves(M);
    const float sc = fast_exp2(m_run[g] - M);
    float l = l_run[g] * sc;
    if constexpr (LPR == 8) l += dpp_ror8(l);
    if constexpr (LPR <= 16) l = sum_row_pairs(l);
    l = sum_halves(l);
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x[e] = acc[g][e] * sc;
      if constexpr (LPR == 8) x[e] += dpp_ror8(x[e]);  // the two groups of a 16-lane row
    }
    float y[4];  // lanes 0-31: values 0 .. 3, lanes 32-63: values 4 .. 7
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = swap_halves_add(x[e], x[e + 4]);
    if constexpr (LPR <= 16) {  // even 16-lane rows: the first two of these, odd rows: the last two
      const f32x2_t z = {swap_rows_add(y[0], y[2]), swap_rows_add(y[1], y[3])};
      if (LPR == 16 || (lane & 8) == 0) *(f32x2_t*)&red[wave][g][8 * dc + 4 * (lane >> 5) + 2 * ((lane >> 4) & 1)] = z;
    } else {
      *(f32x4_t*)&red[wave][g][8 * dc + 4 * (lane >> 5)] = f32x4_t{y[0], y[1], y[2], y[3]};
    }
    if (lane == 0) {
      rml[wave][g][0] = M;
      rml[wave][g][1] = l;
    }
  }
  finish_split<D, G, F16, VARIANT>(p, hh, at, lgbuf, red, rml, lgrow, k_begin, k_end);
}

// ---- the same split with both products on the matrix cores --------------------------------------------------------
//
// For quantised stores and for more than four query heads per KV head the kernel above is bound by its vector
// arithmetic (G dot products per loaded pair of values on top of the dequantisation), not by HBM. Here the G heads are
// padded to the 16 columns of v_mfma_f32_16x16x32 and the rows are operands as they come from memory (key_blocks.h).
// What is left for the vector ALU is the dequantisation (3.5
// instructions per element, as the reference rounds) or half an instruction per V element, and the softmax of 16
// head columns per key. The running maximum is one per head (the four lane groups of a head column agree on it), it
// moves lazily as above. Everything after the key loop is shared with the kernel above.
template <int D, int G, int KV, bool VARIANT>
__global__ __launch_bounds__(NTHREADS, D <= 128 ? 2 : 1) void decode_mfma_kernel(const DecodeParams p, const kvx_h2o_args hh) {
  constexpr bool F16 = kv_elem_f16(KV);
  constexpr bool U8 = !kv_is_plain(KV);  // codes + row state (8-bit or 4-bit store)
  using Blocks = KeyBlocks<D, KV, true>;
  using Rows = typename Blocks::Rows;
  constexpr int KJ = Blocks::KJ, DPL = Blocks::DPL, CH = Blocks::CH;
  constexpr int LGK = logit_floats(G, D, U8) / G;
  __shared__ __align__(16) float lgbuf[LGK * G];  // [key][head]
  __shared__ __align__(16) float red[WAVES][G][D];
  __shared__ float rml[WAVES][G][2];
  static_assert(D == 64 || D == 128 || (D == 256 && U8), "plain rows of 256 values take the vector-ALU kernel");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int m = lane & 15, kg = lane >> 4;
  const int split = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
  const int k_begin = split * p.keys_per_split;
  const int k_end = min(k_begin + p.keys_per_split, p.kv_len);

  u32x4_t qb[KJ];  // B operands of the first product: head m (zero beyond the group), d slice of lane group kg
#pragma unroll
  for (int e = 0; e < KJ; ++e) {
    qb[e] = u32x4_t{0u, 0u, 0u, 0u};
    if (m < p.Gr) qb[e] = *(const u32x4_t*)(p.q + b * p.q_sb + (int64_t)(kvh * p.Gr + m) * p.q_sh + Blocks::kslice(e, kg));
  }
  Blocks blocks;
  blocks.init(p.k, p.v, p.k_scale, p.k_zp, p.v_scale, p.v_zp, b * p.k_sb + kvh * p.k_sh, b * p.v_sb + kvh * p.v_sh, b * p.qs_sb + kvh * p.qs_sh, p.k_st, p.v_st,
              p.qs_vec, m, kg, k_end);
  float* lgrow = p.logits ? p.logits + ((int64_t)b * p.Hkv + kvh) * p.Tpad * G : nullptr;
  int lg_base = k_begin;

  f32x4_t acc[DPL];
#pragma unroll
  for (int t = 0; t < DPL; ++t) acc[t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  float m_run = kNegBig, l_run = 0.0f;

  auto consume = [&](Rows& r, int chunk0) {
    f32x4_t s[2];
#pragma unroll
    for (int gi = 0; gi < 2; ++gi) {
      s[gi] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int e = 0; e < KJ; ++e) s[gi] = mfma_16x16x32<F16>(Blocks::k_operand(r, gi, e), qb[e], s[gi]);
    }
    // this lane: head m, keys chunk0 + 16 gi + 4 kg + i (log2 units)
    float sv[8];
#pragma unroll
    for (int gi = 0; gi < 2; ++gi)
#pragma unroll
      for (int i = 0; i < 4; ++i) sv[4 * gi + i] = s[gi][i] * p.c;
    if (chunk0 + CH > k_end) {
#pragma unroll
      for (int gi = 0; gi < 2; ++gi)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (chunk0 + 16 * gi + 4 * kg + i >= k_end) sv[4 * gi + i] = -INFINITY;
    }
    if (lgrow && m < G && chunk0 < k_end) {
      float* dst = lgbuf + (chunk0 - lg_base + 4 * kg) * G + m;
#pragma unroll
      for (int gi = 0; gi < 2; ++gi)
#pragma unroll
        for (int i = 0; i < 4; ++i) dst[(16 * gi + i) * G] = sv[4 * gi + i];
    }
    float mx = sv[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) mx = fmaxf(mx, sv[i]);
    if (__any(mx > m_run + kRescaleSlack)) {
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));  // the head's maximum over the four lane groups
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float mn = fmaxf(m_run, mx);
      const float al = fast_exp2(m_run - mn);
      m_run = mn;
      l_run *= al;
#pragma unroll
      for (int t = 0; t < DPL; ++t) acc[t] *= al;
    }
    float pv[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      pv[i] = fast_exp2(sv[i] - m_run);
      l_run += pv[i];
    }
    const u32x4_t pb = {pack_pair<F16>(pv[0], pv[1]), pack_pair<F16>(pv[2], pv[3]), pack_pair<F16>(pv[4], pv[5]), pack_pair<F16>(pv[6], pv[7])};
#pragma unroll
    for (int t = 0; t < DPL; ++t) acc[t] = mfma_16x16x32<F16>(Blocks::v_operand(r, t), pb, acc[t]);
  };

  // Two steps in flight per wavefront: the loads of step i + 1 are issued before step i is consumed.
  const int nsteps = (k_end - k_begin + CH * WAVES - 1) / (CH * WAVES);
  const int stride = CH * WAVES;
  int chunk = k_begin + wave * CH;
  constexpr int FLUSH_STEPS = LGK / (CH * WAVES);
  static_assert(LGK % (CH * WAVES) == 0 && FLUSH_STEPS >= 2 && FLUSH_STEPS % 2 == 0, "the loop below advances two steps at a time");
  Rows ra, rb;
  blocks.issue(ra, chunk);
  const RowAt at = row_at<D>(p, hh, b, kvh);
  for (int i = 0; i + 1 < nsteps; i += 2) {
    blocks.issue(rb, chunk + stride);
    __builtin_amdgcn_sched_barrier(0);
    consume(ra, chunk);
    __builtin_amdgcn_sched_barrier(0);  // the loads below reuse the registers consumed above
    blocks.issue(ra, chunk + 2 * stride);
    __builtin_amdgcn_sched_barrier(0);
    consume(rb, chunk + stride);
    __builtin_amdgcn_sched_barrier(0);
    chunk += 2 * stride;
    if (lgrow && !p.resident && ((i + 2) % FLUSH_STEPS == 0 || i + 2 >= nsteps)) {
      __syncthreads();
      flush_logits<G, LGK, CH>(lgbuf, lgrow, lg_base, k_end, tid);
      lg_base += LGK;
      __syncthreads();
    }
  }
  // the last of an odd number of steps on its own: with the loads and the work of a second one, splits of one step took 1 us longer.
  // Out of line: an even number of steps goes on without fetching past it.
  if (__builtin_expect(nsteps & 1, 0)) {
    consume(ra, chunk);
    if (lgrow && !p.resident) {
      __syncthreads();
      flush_logits<G, LGK, CH>(lgbuf, lgrow, lg_base, k_end, tid);
    }
  }

  // ---- this wavefront's partial: sums over the four lane groups of a head, outputs by d ----------------------------
  float l = l_run;
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (m < G) {
#pragma unroll
    for (int t = 0; t < DPL; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[wave][m][Blocks::dmap(t, 4 * kg + i)] = acc[t][i];
    if (kg == 0) {
      rml[wave][m][0] = m_run;
      rml[wave][m][1] = l;
    }
  }
  finish_split<D, G, F16, VARIANT>(p, hh, at, lgbuf, red, rml, lgrow, k_begin, k_end);
}

// Combine the splits of one (b, query head): 4 groups of D threads each take a quarter of the
// splits, then the groups are added through LDS. Its first wavefront also produces the base-2 log-sum-exp.
template <int D, bool F16>
__device__ __forceinline__ void merge_job(const DecodeParams& p, const int bh) {
  __shared__ float red[4][D + 1];
  __shared__ float sM;
  const int b = bh / p.Hq, hqi = bh % p.Hq;
  const int d = threadIdx.x % D, grp = threadIdx.x / D;
  const float* ml = p.part_ml + (int64_t)bh * p.num_splits * 2;
  if (threadIdx.x < 64) {
    float mloc = -INFINITY;
    for (int s = threadIdx.x; s < p.num_splits; s += 64) mloc = fmaxf(mloc, ml[2 * s]);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) mloc = fmaxf(mloc, __shfl_xor(mloc, off, 64));
    if (threadIdx.x == 0) sM = mloc;
    // the log-sum-exp by the routine the split kernel uses for its own weights: the same bits on either route
    const float lse = row_sum(ml, p.num_splits, threadIdx.x).lse();
    if (threadIdx.x == 0 && p.lse_out) p.lse_out[bh] = lse;
  }
  __syncthreads();
  const float M = sM;
  float L = 0.0f, acc = 0.0f;
  for (int s = grp; s < p.num_splits; s += 4) {
    const float w = fast_exp2(ml[2 * s] - M);
    L += ml[2 * s + 1] * w;
    acc += p.part_o[(((int64_t)(bh / p.Gr) * p.num_splits + s) * p.Gr + bh % p.Gr) * D + d] * w;
  }
  red[grp][d] = acc;
  if (d == 0) red[grp][D] = L;
  __syncthreads();
  if (grp == 0) {
    const float a4 = red[0][d] + red[1][d] + red[2][d] + red[3][d];
    const float l4 = red[0][D] + red[1][D] + red[2][D] + red[3][D];
    const float r = a4 / l4;
    const float other = __shfl_xor(r, 1, 64);
    if ((d & 1) == 0) *(uint32_t*)(p.o + b * p.o_sb + hqi * p.o_sh + d) = pack_pair<F16>(r, other);
  }
}

// W[b, kvh, k] = (1/G) sum_g exp2(logit[b, kvh, k, g] - lse[b, kvh*G+g]); one key per lane and pass,
// 4096 keys per workgroup of NT threads, where the logits went to the scratch. With H2O set it also does the cache's score update and eviction choice
// in the same pass (keys_values/kvcache/h2o.py:175-196, keys_values/kvcache/attn_weights.py:773-774
// for one slot): scores += W, then the (value, slot) minimum of the row through an integer atomicMin; the workgroup
// that finishes last publishes the slot of every row's minimum. (That needs no fence: the minima and the count of
// finished workgroups are device-scope atomics, each waited for before the next; a release fence per workgroup
// would write the whole L2 back on this multi-die part.)
template <int G, bool H2O, int NT>
__device__ __forceinline__ void weights_job(const DecodeParams& p, const kvx_h2o_args& hh, const int bx, const int kvh, const int b, const int jobs) {
  typedef float fG __attribute__((ext_vector_type(G >= 4 ? 4 : (G == 2 ? 2 : 1))));
  constexpr int NV = G >= 4 ? G / 4 : 1;
  constexpr int PASSES = 4096 / NT;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  __shared__ float lse_sh[G];
  __shared__ unsigned long long wbest[NT / 64];
  __shared__ int last_job;
  unsigned long long mine = ~0ull;
  {
    // the row's log-sum-exps from the splits' partials, by the routine the split kernel and the merge use
    for (int g = wave; g < G; g += NT / 64) {
      float l = INFINITY;  // dummy heads: exp2(x - inf) = 0
      if (g < p.Gr) l = row_sum(p.part_ml + ((int64_t)b * p.Hq + kvh * p.Gr + g) * p.num_splits * 2, p.num_splits, lane).lse();
      if (lane == 0) lse_sh[g] = l;
    }
    __syncthreads();
    float lse[G];
#pragma unroll
    for (int g = 0; g < G; ++g) lse[g] = lse_sh[g];
    const float* lgrow = p.logits + ((int64_t)b * p.Hkv + kvh) * p.Tpad * G;
    float* wr = p.w ? p.w + ((int64_t)b * p.Hkv + kvh) * p.kv_len : nullptr;
    float* sc = H2O ? hh.scores + b * hh.sc_stride_b + kvh * hh.sc_stride_h : nullptr;
    const int32_t* tpr = (H2O && hh.token_pos) ? hh.token_pos + b * hh.tp_stride_b + kvh * hh.tp_stride_h : nullptr;
    fG t[PASSES][NV];
#pragma unroll
    for (int it = 0; it < PASSES; ++it) {
      const int k = min(bx * 4096 + it * NT + tid, p.Tpad - 1);
#pragma unroll
      for (int j = 0; j < NV; ++j) t[it][j] = *((const fG*)(lgrow + (int64_t)k * G) + j);
    }
#pragma unroll
    for (int it = 0; it < PASSES; ++it) {
      const int k = bx * 4096 + it * NT + tid;
      if (k >= p.kv_len) break;
      float acc = 0.0f;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float x;
        if constexpr (G >= 4) x = t[it][g / 4][g % 4];
        else if constexpr (G == 2) x = t[it][0][g];
        else x = t[it][0][0];
        acc += fast_exp2(x - lse[g]);
      }
      acc *= 1.0f / (float)p.Gr;
      if (wr) wr[k] = acc;
      if constexpr (H2O) {
        float val = sc[k] + acc;
        sc[k] = val;
        if (k < hh.limit) {
          if (hh.normalize) val = val / (float)(hh.input_pos - max(tpr[k], hh.prefill_len - 1));
          const unsigned long long key = ((unsigned long long)ordered_bits(val) << 32) | (unsigned)k;
          mine = key < mine ? key : mine;
        }
      }
    }
  }
  if constexpr (H2O) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      const unsigned long long o = __shfl_xor(mine, off, 64);
      mine = o < mine ? o : mine;
    }
    if (lane == 0) wbest[wave] = mine;
    __syncthreads();
    if (tid == 0) {
      unsigned long long mn = wbest[0];
      for (int i = 1; i < NT / 64; ++i) mn = wbest[i] < mn ? wbest[i] : mn;
      if (mn != ~0ull) {
        const unsigned long long old = __hip_atomic_fetch_min(p.best + b * p.Hkv + kvh, mn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" : : "v"(old) : "memory");  // performed before this workgroup counts itself
      }
      // counted per row first, rows second: no counter sees more than a few dozen increments
      const int wx = jobs / (p.B * p.Hkv);
      const uint32_t row_full = (uint32_t)wx - 1u;
      const bool row_last = __hip_atomic_fetch_add(p.row_count + (b * p.Hkv + kvh) * kCountStride, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == row_full;
      last_job = row_last && __hip_atomic_fetch_add(p.tail_count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)(p.B * p.Hkv - 1);
    }
    __syncthreads();
    if (last_job) {
      for (int i = tid; i < p.B * p.Hkv; i += NT)
        hh.next_index[i] = (int32_t)(__hip_atomic_load(p.best + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 0xffffffffull);
    }
  }
}

// What follows the split kernel where the logits go through the scratch by plan, in one launch: the first merge_jobs workgroups combine the splits of one (batch,
// query head) each; the others (MODE 1: weights wanted, MODE 2: fused H2O step) take 4096 keys of a (batch, KV head)
// row each. The two kinds do not depend on each other: both read what the split kernel left.
template <int D, bool F16, int G, int MODE>
__global__ __launch_bounds__(4 * D) void decode_tail_kernel(const DecodeParams p, const kvx_h2o_args hh, const int merge_jobs, const int wx) {
  if ((int)blockIdx.x < merge_jobs) {
    merge_job<D, F16>(p, blockIdx.x);
    return;
  }
  const int j = blockIdx.x - merge_jobs;
  weights_job<G, MODE == 2, 4 * D>(p, hh, j % wx, (j / wx) % p.Hkv, j / (wx * p.Hkv), (int)gridDim.x - merge_jobs);
}

template <int D, bool F16, int G>
int launch_tail(const DecodeParams& p, const kvx_h2o_args* hh, hipStream_t st) {
  const int merge_jobs = p.B * p.Hq, wx = (p.kv_len + 4095) / 4096;
  const int weight_jobs = hh || p.w ? wx * p.Hkv * p.B : 0;
  const dim3 grid(merge_jobs + weight_jobs), block(4 * D);
  const kvx_h2o_args h2 = hh ? *hh : kvx_h2o_args{};
  if (hh) hipLaunchKernelGGL((decode_tail_kernel<D, F16, G, 2>), grid, block, 0, st, p, h2, merge_jobs, wx);
  else hipLaunchKernelGGL((decode_tail_kernel<D, F16, G, 1>), grid, block, 0, st, p, h2, merge_jobs, wx);
  KVX_HIP(hipGetLastError());
  return KVX_OK;
}

// The split kernel and, where the logits go through the scratch by plan, the tail.
template <int D, int G>
int launch_dg(const DecodeParams& p, int kv, const kvx_h2o_args* hh, hipStream_t st) {
  dim3 grid(p.num_splits, p.Hkv, p.B);
  const kvx_h2o_args h2 = hh ? *hh : kvx_h2o_args{};
  // quantised stores and groups of 8 heads or more: both products on the matrix cores
  auto launch = [&](auto kv_tag) {
    constexpr int KV = decltype(kv_tag)::value;
    constexpr bool MFMA = !kv_is_plain(KV) || (D <= 128 && G >= 8);
    const bool variant = hh && (hh->v_norm || hh->q_errors);
    if constexpr (MFMA) {
      if (variant) hipLaunchKernelGGL((decode_mfma_kernel<D, G, KV, true>), grid, dim3(NTHREADS), 0, st, p, h2);
      else hipLaunchKernelGGL((decode_mfma_kernel<D, G, KV, false>), grid, dim3(NTHREADS), 0, st, p, h2);
    } else if constexpr (G <= 8) {
      if (variant) hipLaunchKernelGGL((decode_split_kernel<D, G, KV, true>), grid, dim3(NTHREADS), 0, st, p, h2);
      else hipLaunchKernelGGL((decode_split_kernel<D, G, KV, false>), grid, dim3(NTHREADS), 0, st, p, h2);
    }
  };
  switch (kv) {
#define KVX_DECODE_CASE(KV) case KV: launch(std::integral_constant<int, KV>{}); break;
    KVX_DECODE_CASE(KVX_KV_BF16)
    KVX_DECODE_CASE(KVX_KV_F16)
    KVX_DECODE_CASE(KVX_KV_U8)
    KVX_DECODE_CASE(KVX_KV_U4)
    KVX_DECODE_CASE(KVX_KV_U8_F16)
    KVX_DECODE_CASE(KVX_KV_U4_F16)
#undef KVX_DECODE_CASE
  }
  KVX_HIP(hipGetLastError());
  if (p.one_launch) return KVX_OK;
  return kv_elem_f16(kv) ? launch_tail<D, true, G>(p, hh, st) : launch_tail<D, false, G>(p, hh, st);
}

template <int D>
int launch_d(const DecodeParams& p, int G, int kv, const kvx_h2o_args* hh, hipStream_t st) {
  switch (G) {
    case 1: return launch_dg<D, 1>(p, kv, hh, st);
    case 2: return launch_dg<D, 2>(p, kv, hh, st);
    case 4: return launch_dg<D, 4>(p, kv, hh, st);
    case 8: return launch_dg<D, 8>(p, kv, hh, st);
    case 16:
      if constexpr (D <= 128) return launch_dg<D, 16>(p, kv, hh, st);
      break;
  }
  return set_error(KVX_ERR_UNSUPPORTED, "kvx_sdpa_decode: %d query heads per KV head (at most 16; at most 8 with head size 256)", p.Gr);
}

}  // namespace decode

// one per head size, each in a file of its own
int launch_decode_64(const decode::DecodeParams& p, int G, int kv, const kvx_h2o_args* hh, hipStream_t st);
int launch_decode_128(const decode::DecodeParams& p, int G, int kv, const kvx_h2o_args* hh, hipStream_t st);
int launch_decode_256(const decode::DecodeParams& p, int G, int kv, const kvx_h2o_args* hh, hipStream_t st);

}  // namespace kvx
