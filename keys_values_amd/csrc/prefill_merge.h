// The combination of the attention kernel's per-split partials, as a job of one workgroup: the combining kernel
// (sdpa_prefill.hip) runs it alone, the score-sum kernel of short chunks (score_sum.hip) beside its own work.
#pragma once
#include "kvx_common.h"

namespace kvx {

struct MergeParams {
  const float* part_o;   // [split][group][R][D] fp32, unnormalised
  const float* part_ml;  // [split][team][group][R][2]  (max in log2 units, sum)
  uint16_t* o;
  float* lse;  // (B, q_len, Hq) or NULL
  int32_t B, Hq, Hkv, G, q_len, R, num_splits;
  int64_t o_sb, o_sh, o_st;
  int32_t input_pos, split_keys;  // slots in position order: keys of a split; a row has no partial in splits behind its position. 0: all splits
  int32_t teams;  // 1, or 2 where a split's partial is of two teams (relative to the larger of their maxima): the sums are added as if of two splits
};

// Combine the per-split partials of a row: D / 4 threads a row, each four values, times SC split classes that take
// splits j, j + SC, ... and are added through LDS. Bound by HBM (every partial is read once) where there are many rows;
// with few rows (32 queries over 32768 keys: 1024 rows of 32 splits) a thread's walk over the splits was the time, a memory
// latency per split and 15 us of a 46 us call: four loads in flight and SC classes make it about two latencies.
// The first four partials are asked for together with their maxima, and up to four splits the maxima are read once: 32768 rows of 2 splits of
// 128 values 11.3 -> 9.4 us (4.6 TB/s), 24000 of 2 to 3 of 256 14.0 -> 11.4, 960 of 16 of 64 7.2 -> 5.9.
// ROWS: rows of one workgroup of 256 threads.
constexpr int merge_rows(int D, int SC) { return 256 / (D / 4 * SC); }  // D: 64, 128 or 256
// split classes while a walk is longer than four splits and the rows alone leave the device short of threads
constexpr int merge_classes(int D) { return 256 / (D / 4) < 8 ? 256 / (D / 4) : 8; }
inline bool merge_wants_classes(const MergeParams& p, int D) {
  return p.num_splits > 4 && (int64_t)p.B * p.Hkv * p.R * (D / 4) < (int64_t)num_cus() * 256;
}
// Where a (batch, KV head) pair has many blocks of rows, they go round the pairs: pair g's on the die (of eight, which take workgroups in turn) whose
// L2 cache the attention kernel's workgroups of g have written. Rows in order -> round the pairs, calls without weights, us: 294 rows over 16 x 1996 keys of 128
// 21.7 -> 19.0, 214 of 256 over 8 x 1127 25.4 -> 20.6, 1716 of 64 over 8 x 1800 19.5 -> 17.6. Partials that do not fit the dies' 8 x 4 MB come from memory, in
// order the faster: 1597 tokens of 16 heads of 256 over 8 58.7, round the pairs 59.7.
__host__ __device__ inline bool merge_by_pair(const MergeParams& p, int D, int rows) {
  return p.R >= 8 * rows && (int64_t)p.num_splits * p.B * p.Hkv * p.R * D <= (8 << 20);
}
inline int64_t merge_blocks(const MergeParams& p, int D, int SC) {
  const int rows = merge_rows(D, SC);
  const int64_t pairs = (int64_t)p.B * p.Hkv;
  return merge_by_pair(p, D, rows) ? pairs * ((p.R + rows - 1) / rows) : (pairs * p.R + rows - 1) / rows;
}
template <int D, bool F16, int SC, int TEAMS>
__device__ __forceinline__ void merge_rows_job(const MergeParams& p, const int64_t block, const int tid, f32x4_t* red_o, float* red_l) {
  constexpr int TPR = D / 4;                // threads per row and split class
  constexpr int ROWS = merge_rows(D, SC);    // rows per workgroup
  static_assert(ROWS >= 1, "a row's threads fit a workgroup");
  const int64_t total_rows = (int64_t)p.B * p.Hkv * p.R;
  int64_t grow = block * ROWS + tid / (TPR * SC);
  bool live = grow < total_rows;
  if (merge_by_pair(p, D, ROWS)) {
    const uint32_t pairs = (uint32_t)(p.B * p.Hkv), at = (uint32_t)block / pairs;
    const int row = (int)at * ROWS + tid / (TPR * SC);
    live = row < p.R;
    grow = (int64_t)((uint32_t)block - at * pairs) * p.R + row;
  }
  const int64_t growc = live ? grow : total_rows - 1;
  const int S = p.split_keys ? min(p.num_splits, (p.input_pos + (int)(growc % p.R) / p.G) / p.split_keys + 1) : p.num_splits;
  const int dq = tid % TPR, j = (tid / TPR) % SC;
  const f32x2_t* ml = (const f32x2_t*)p.part_ml + growc;  // (maximum, sum) of split s at s * TEAMS * total_rows, of its second team behind it
  const float* po = p.part_o + growc * D + dq * 4;
  // the partials of splits s0, s0 + SC, ... (four at most), all asked for at once; nothing where there is no such split
  f32x2_t m[4], m2[4];
  f32x4_t x[4];
  auto load = [&](int s0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      m[u] = m2[u] = f32x2_t{-INFINITY, 0.0f};
      x[u] = f32x4_t{0, 0, 0, 0};
      if (s0 + u * SC < S) {
        const int64_t at = (int64_t)(s0 + u * SC) * total_rows;
        m[u] = ml[at * TEAMS];
        if constexpr (TEAMS > 1) m2[u] = ml[at * TEAMS + total_rows];
        x[u] = *(const f32x4_t*)(po + at * D);
      }
    }
  };
  load(j);
  float M;
  if (SC == 1 && S <= 4) {
    M = -INFINITY;
#pragma unroll
    for (int u = 0; u < 4; ++u) M = fmaxf(M, TEAMS > 1 ? fmaxf(m[u][0], m2[u][0]) : m[u][0]);
  } else {
    M = -INFINITY;
    // a lane each; every thread reading them all was two thirds of the launch (1976 rows of 18 maxima 12 us)
    for (int i = dq; i < S * TEAMS; i += TPR) M = fmaxf(M, ml[(int64_t)i * total_rows][0]);
#pragma unroll
    for (int off = TPR / 2; off >= 1; off >>= 1) M = fmaxf(M, __shfl_xor(M, off, 64));
  }
  const float Mu = (M == -INFINITY) ? 0.0f : M;
  float L = 0.0f;
  f32x4_t acc = {0, 0, 0, 0};
  for (int s0 = j; s0 < S; s0 += 4 * SC) {
    if (s0 != j) load(s0);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (s0 + u * SC < S) {
        float w = fast_exp2(m[u][0] - Mu);
        L += m[u][1] * w;
        if constexpr (TEAMS > 1) {
          const float w2 = fast_exp2(m2[u][0] - Mu);
          L += m2[u][1] * w2;
          w = fmaxf(w, w2);
        }
        acc += x[u] * w;
      }
  }
  if constexpr (SC > 1) {
    red_o[tid] = acc;
    red_l[tid] = L;
    __syncthreads();
    if (j != 0) return;
#pragma unroll
    for (int i = 1; i < SC; ++i) {
      acc += red_o[tid + i * TPR];
      L += red_l[tid + i * TPR];
    }
  }
  if (!live) return;
  const int group = (int)(grow / p.R);
  const int row = (int)(grow % p.R);
  const int b = group / p.Hkv, kvh = group % p.Hkv;
  const int qi = row / p.G, g = row % p.G;
  const float inv = L > 0.0f ? 1.0f / L : 0.0f;
  uint16_t* op = p.o + b * p.o_sb + (int64_t)(kvh * p.G + g) * p.o_sh + (int64_t)qi * p.o_st + dq * 4;
  u32x2_t w2;
  w2[0] = pack_pair<F16>(acc[0] * inv, acc[1] * inv);
  w2[1] = pack_pair<F16>(acc[2] * inv, acc[3] * inv);
  *(u32x2_t*)op = w2;
  if (p.lse && dq == 0) p.lse[((int64_t)b * p.q_len + qi) * p.Hq + kvh * p.G + g] = Mu + fast_log2(L);
}

// tid: the thread's place among the 256 of the job (SC > 1: of the workgroup)
template <int D, bool F16, int SC>
__device__ __forceinline__ void merge_job(const MergeParams& p, const int64_t block, const int tid) {
  __shared__ f32x4_t red_o[SC > 1 ? 256 : 1];
  __shared__ float red_l[SC > 1 ? 256 : 1];
  if (p.teams > 1) merge_rows_job<D, F16, SC, 2>(p, block, tid, red_o, red_l);
  else merge_rows_job<D, F16, SC, 1>(p, block, tid, red_o, red_l);
}

}  // namespace kvx
