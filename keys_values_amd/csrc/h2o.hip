// H2O score update and eviction choice for gfx950.
//
// Reference behaviour: keys_values/kvcache/h2o.py:146-199 (scores += weights, optional
// normalisation by residency) and keys_values/kvcache/attn_weights.py:771-783 (argsort / topk of
// the smallest scores). Output order here is ascending (value, slot), i.e. a stable argsort cut at k.
//
// Two shapes of the problem:
//   k == 1 (single-token decode): a streaming pass over all rows with many workgroups; each folds
//          its slice into one 64-bit key (ordered value bits << 32 | slot) and publishes it with
//          an integer atomicMin, which is order independent and therefore deterministic.
//   k  > 1 (chunked prefill): a row is spread over workgroups of 256, 512 or 1024 slots. The first launch adds the weights
//          and sorts every workgroup's 64-bit (value, slot) keys; the second gives every key that can be among
//          the first k its rank in the row by binary searches in the other lists and writes it there.
//          Without the workspace for the lists (one workgroup per row): the first pass adds the weights and
//          leaves the row's ordered value bits in LDS (rows of up to ~36K slots; longer rows are
//          re-read from global memory). A 4-pass 8-bit radix select finds the k-th smallest value;
//          elements below it, plus the lowest-slot elements equal to it, are gathered and
//          bitonic-sorted as 64-bit (value, slot) keys.
#include <mutex>
#include <type_traits>

#include "kvx_common.h"

namespace kvx {
namespace {


// Monotone map float -> uint32 (a < b  <=>  key(a) < key(b)); -0.0 is folded onto +0.0 first, as
// comparisons treat them as equal.
__device__ __forceinline__ uint32_t ordered_bits(float x) {
  x += 0.0f;
  const uint32_t u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Value the selection compares: the score, or the score divided by the slot's residency
// (keys_values/kvcache/h2o.py:183-196).
__device__ __forceinline__ float residency_of(float score, const kvx_h2o_args& a, int position) {  // (of a slot's token)
  if (!a.normalize) return score;
  return score / (float)(a.input_pos - max(position, a.prefill_len - 1));
}
__device__ __forceinline__ float residency_value(float score, const kvx_h2o_args& a, const int32_t* tp_row, int idx) {
  return residency_of(score, a, a.normalize ? tp_row[idx] : 0);
}

// Q-Hitter combination (keys_values/kvcache/qh2o.py:178-210): both terms are min-max normalised over
// all (head, slot < limit) entries of the batch element, then c*s + ((c-1)/2)*q + (1-c). Each
// product and sum is rounded on its own, as the reference's tensor expression is.
struct Modify {
  const float* qe;  // q_errors row, or nullptr: no modification
  float smin, sden, qmin, qden;
  float c, c2, c3;
};

// stats: 4 floats per (batch, head) row = min / max of the compared value and of q_errors.
__device__ __forceinline__ Modify load_modify(const kvx_h2o_args& a, const float* stats, int b, int hh) {
  Modify m;
  m.qe = nullptr;
  if (!stats) return m;
  m.qe = a.q_errors + b * a.sc_stride_b + hh * a.sc_stride_h;
  float smin = INFINITY, smax = -INFINITY, qmin = INFINITY, qmax = -INFINITY;
  for (int h = 0; h < a.Hkv; ++h) {
    const f32x4_t st = *(const f32x4_t*)(stats + ((int64_t)b * a.Hkv + h) * 4);
    smin = fminf(smin, st[0]);
    smax = fmaxf(smax, st[1]);
    qmin = fminf(qmin, st[2]);
    qmax = fmaxf(qmax, st[3]);
  }
  m.smin = smin;
  m.sden = smax - smin;
  m.qmin = qmin;
  m.qden = qmax - qmin;
  m.c = (float)a.combination;
  m.c2 = (float)((a.combination - 1.0) / 2.0);
  m.c3 = (float)(1.0 - a.combination);
  return m;
}

__device__ __forceinline__ float combined_value(float v, float qerr, const Modify& m) {
  const float s = (v - m.smin) / m.sden;
  const float q = (qerr - m.qmin) / m.qden;
  return __fadd_rn(__fadd_rn(__fmul_rn(m.c, s), __fmul_rn(m.c2, q)), m.c3);
}

__device__ __forceinline__ float select_value(float score, const kvx_h2o_args& a, const int32_t* tp_row, int idx, const Modify& m) {
  const float v = residency_value(score, a, tp_row, idx);
  return m.qe ? combined_value(v, m.qe[idx], m) : v;
}

// ---- policy variants: the accumulation pass ---------------------------------------------------

constexpr int SEL_THREADS = 1024;

// Deterministic workgroup reductions (wavefront butterfly, then the 16 partials in a fixed order).
template <int THREADS = SEL_THREADS, typename Op>
__device__ __forceinline__ float block_reduce(float v, float* red, Op op) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = op(v, __shfl_xor(v, off, 64));
  __syncthreads();  // red may still be read from the previous reduction
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float r = red[0];
  for (int i = 1; i < THREADS / 64; ++i) r = op(r, red[i]);
  return r;
}

// The value of the lane whose index differs in bit log2(S), on the vector ALU.
template <int S>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
  auto dpp = [](uint32_t x, auto ctrl) { return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, decltype(ctrl)::value, 0xf, 0xf, true); };
  if constexpr (S == 1) return dpp(v, std::integral_constant<int, 0xB1>{});        // quad_perm [1,0,3,2]
  else if constexpr (S == 2) return dpp(v, std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
  else if constexpr (S == 4) return dpp(dpp(v, std::integral_constant<int, 0x141>{}), std::integral_constant<int, 0x1B>{});  // half mirror, quad mirror
  else if constexpr (S == 8) return dpp(v, std::integral_constant<int, 0x128>{});  // row_ror:8
  else if constexpr (S == 16) {
    const u32pair_t r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return (threadIdx.x & 16) ? r[0] : r[1];
  } else {
    const u32pair_t r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return (threadIdx.x & 32) ? r[0] : r[1];
  }
}

// Least, largest, least and largest of a workgroup's four values in one exchange: four reductions one after the other took a third of the launches that
// need them (16 rows of 6000 slots, us: statistics 8.2 -> 7.3, sort 6.3 -> 5.5). Called once by a kernel. AT_ONCE: wavefronts whose
// values are read together; all 16 of 1024 threads are 60 registers, with which the sort of 1024 keys left a unit room for one workgroup, not two
// (20 choices of 1 to 32 rows of 37000 to 115000 slots: 39.2 us in the mean, 48.1 that way).
template <int THREADS, int AT_ONCE = THREADS / 64>
__device__ __forceinline__ f32x4_t block_extremes(f32x4_t v) {
  __shared__ f32x4_t red[THREADS / 64];
  auto fold = [](const f32x4_t& x, const f32x4_t& y) { return f32x4_t{fminf(x[0], y[0]), fmaxf(x[1], y[1]), fminf(x[2], y[2]), fmaxf(x[3], y[3])}; };
  auto lanes = [&](auto s_tag) {
    constexpr int S = decltype(s_tag)::value;
    f32x4_t o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = __uint_as_float(lane_xor<S>(__float_as_uint(v[i])));
    v = fold(v, o);
  };
  lanes(std::integral_constant<int, 32>{});
  lanes(std::integral_constant<int, 16>{});
  lanes(std::integral_constant<int, 8>{});
  lanes(std::integral_constant<int, 4>{});
  lanes(std::integral_constant<int, 2>{});
  lanes(std::integral_constant<int, 1>{});
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  f32x4_t r = red[0];
#pragma unroll AT_ONCE
  for (int i = 1; i < THREADS / 64; ++i) r = fold(r, red[i]);
  return r;
}

// One workgroup per (batch, head) row: scores += instantaneous score, where the latter is w or,
// with v_norm, (v_norm*w / sum(v_norm*w)) * q_len (keys_values/kvcache/h2o.py:297-314); and the row's
// min / max of the compared value and of q_errors over the slots below limit, for the combination.
__global__ __launch_bounds__(SEL_THREADS) void accumulate_kernel(const kvx_h2o_args a, float* __restrict__ stats) {
  __shared__ float red[SEL_THREADS / 64];
  const int tid = threadIdx.x;
  const int row = blockIdx.x;
  const int b = row / a.Hkv, hh = row % a.Hkv;
  const int64_t off = b * a.sc_stride_b + hh * a.sc_stride_h;
  float* sc = a.scores + off;
  const float* w = a.w ? a.w + (int64_t)row * a.kv_len : nullptr;
  const float* vn = a.v_norm ? a.v_norm + off : nullptr;
  const float* qe = a.q_errors ? a.q_errors + off : nullptr;
  const int32_t* tpr = a.token_pos ? a.token_pos + b * a.tp_stride_b + hh * a.tp_stride_h : nullptr;
  float z = 1.0f;
  if (w && vn) {
    float part = 0.0f;
    for (int i = tid; i < a.kv_len; i += SEL_THREADS) part += vn[i] * w[i];
    z = block_reduce(part, red, [](float x, float y) { return x + y; });
  }
  const float ql = (float)a.q_len;
  float smin = INFINITY, smax = -INFINITY, qmin = INFINITY, qmax = -INFINITY;
  constexpr int PB = 4;
  for (int i0 = tid; i0 < a.kv_len; i0 += PB * SEL_THREADS) {
    float sv[PB], wv[PB], nv[PB], qv[PB];
#pragma unroll
    for (int j = 0; j < PB; ++j) {  // all loads of the batch before the first store (sc may alias for all the compiler knows)
      const int i = i0 + j * SEL_THREADS;
      const bool in = i < a.kv_len;
      sv[j] = in ? sc[i] : 0.0f;
      wv[j] = (in && w) ? w[i] : 0.0f;
      nv[j] = (in && w && vn) ? vn[i] : 0.0f;
      qv[j] = (qe && i < a.limit) ? qe[i] : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < PB; ++j) {
      const int i = i0 + j * SEL_THREADS;
      if (i >= a.kv_len) break;
      float v = sv[j];
      if (w) {
        float inst = wv[j];
        if (vn) inst = __fmul_rn(__fmul_rn(nv[j], wv[j]) / z, ql);
        v = __fadd_rn(v, inst);
        sc[i] = v;
      }
      if (qe && i < a.limit) {
        const float cv = residency_value(v, a, tpr, i);
        smin = fminf(smin, cv);
        smax = fmaxf(smax, cv);
        qmin = fminf(qmin, qv[j]);
        qmax = fmaxf(qmax, qv[j]);
      }
    }
  }
  if (qe) {
    const f32x4_t x = block_extremes<SEL_THREADS>(f32x4_t{smin, smax, qmin, qmax});
    if (tid == 0) *(f32x4_t*)(stats + (int64_t)row * 4) = x;
  }
}

// ---- k == 1 ---------------------------------------------------------------------------------

__global__ void argmin_init_kernel(unsigned long long* best, int rows) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < rows) best[i] = ~0ull;
}

__global__ __launch_bounds__(256) void update_argmin_kernel(const kvx_h2o_args a, unsigned long long* best, const float* stats) {
  const int row = blockIdx.y;
  const int b = row / a.Hkv, hh = row % a.Hkv;
  const Modify md = load_modify(a, stats, b, hh);
  float* sc = a.scores + b * a.sc_stride_b + hh * a.sc_stride_h;
  const float* w = a.w ? a.w + (int64_t)row * a.kv_len : nullptr;
  const int32_t* tpr = a.token_pos ? a.token_pos + b * a.tp_stride_b + hh * a.tp_stride_h : nullptr;
  unsigned long long mine = ~0ull;
  // 4 consecutive slots per lane per step, 4096 slots per workgroup
  const int base = blockIdx.x * 4096;
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const int i0 = base + it * 1024 + threadIdx.x * 4;
    // 16-byte loads need 16-byte aligned rows: the score rows by their strides, the rows of w (kv_len long) by kv_len
    if (i0 + 3 < a.kv_len && ((a.sc_stride_h | a.sc_stride_b) & 3) == 0 && (!w || (a.kv_len & 3) == 0)) {
      f32x4_t s = *(const f32x4_t*)(sc + i0);
      if (w) {
        const f32x4_t ww = *(const f32x4_t*)(w + i0);
        s += ww;
        *(f32x4_t*)(sc + i0) = s;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i0 + e < a.limit) {
          const unsigned long long key = ((unsigned long long)ordered_bits(select_value(s[e], a, tpr, i0 + e, md)) << 32) | (unsigned)(i0 + e);
          mine = key < mine ? key : mine;
        }
    } else {
      for (int e = 0; e < 4; ++e) {
        const int i = i0 + e;
        if (i >= a.kv_len) break;
        float s = sc[i];
        if (w) {
          s += w[i];
          sc[i] = s;
        }
        if (i < a.limit) {
          const unsigned long long key = ((unsigned long long)ordered_bits(select_value(s, a, tpr, i, md)) << 32) | (unsigned)i;
          mine = key < mine ? key : mine;
        }
      }
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const unsigned long long o = __shfl_xor(mine, off, 64);
    mine = o < mine ? o : mine;
  }
  __shared__ unsigned long long wbest[4];
  if ((threadIdx.x & 63) == 0) wbest[threadIdx.x >> 6] = mine;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long m = wbest[0];
    for (int i = 1; i < 4; ++i) m = wbest[i] < m ? wbest[i] : m;
    if (m != ~0ull) atomicMin(best + row, m);
  }
}

__global__ void argmin_finish_kernel(const unsigned long long* best, int32_t* next_index, int rows) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < rows) next_index[i] = (int32_t)(best[i] & 0xffffffffull);
}

// ---- k == 1 of a single-token step with the Q-Hitter combination ------------------------------
//
// The scores are up to date and their extremes (and those of the errors) lie in `per_row` records a row; what is left is
// one pass over scores and errors. Workgroups of SEL_ONE slots; the last one of a row (counted in a word the caller zeroed)
// publishes the row's slot. One launch instead of four (statistics, reset, minimum, publication).
constexpr int SEL_ONE = 8 * SEL_THREADS;

__global__ __launch_bounds__(SEL_THREADS) void select_one_kernel(const kvx_h2o_args a, const float* stats, int per_row, uint32_t* counters,
                                                                 unsigned long long* part) {
  __shared__ unsigned long long wbest[SEL_THREADS / 64];
  __shared__ uint32_t last;
  const int tid = threadIdx.x, row = blockIdx.y, b = row / a.Hkv, hh = row % a.Hkv;
  float v4[4] = {INFINITY, -INFINITY, INFINITY, -INFINITY};
  const float* st = stats + (int64_t)b * a.Hkv * per_row * 4;
  for (int i = tid; i < a.Hkv * per_row; i += SEL_THREADS) {
    const f32x4_t s = *(const f32x4_t*)(st + i * 4);
    v4[0] = fminf(v4[0], s[0]);
    v4[1] = fmaxf(v4[1], s[1]);
    v4[2] = fminf(v4[2], s[2]);
    v4[3] = fmaxf(v4[3], s[3]);
  }
  const int64_t off = b * a.sc_stride_b + hh * a.sc_stride_h;
  const float *sc = a.scores + off, *qe = a.q_errors + off;
  const int32_t* tpr = a.token_pos ? a.token_pos + b * a.tp_stride_b + hh * a.tp_stride_h : nullptr;
  const int base = blockIdx.x * SEL_ONE + tid;
  float s8[8], q8[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int k = min(base + i * SEL_THREADS, a.limit - 1);
    s8[i] = sc[k];
    q8[i] = qe[k];
  }
  const f32x4_t ex = block_extremes<SEL_THREADS>(f32x4_t{v4[0], v4[1], v4[2], v4[3]});
  Modify m;
  m.qe = qe;
  m.smin = ex[0];
  m.sden = ex[1] - m.smin;
  m.qmin = ex[2];
  m.qden = ex[3] - m.qmin;
  m.c = (float)a.combination;
  m.c2 = (float)((a.combination - 1.0) / 2.0);
  m.c3 = (float)(1.0 - a.combination);
  unsigned long long mine = ~0ull;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int k = base + i * SEL_THREADS;
    if (k >= a.limit) break;
    const unsigned long long key = ((unsigned long long)ordered_bits(combined_value(residency_value(s8[i], a, tpr, k), q8[i], m)) << 32) | (unsigned)k;
    mine = key < mine ? key : mine;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const unsigned long long x = __shfl_xor(mine, o, 64);
    mine = x < mine ? x : mine;
  }
  if ((tid & 63) == 0) wbest[tid >> 6] = mine;
  __syncthreads();
  if (tid != 0) return;
  for (int i = 1; i < SEL_THREADS / 64; ++i) mine = wbest[i] < mine ? wbest[i] : mine;
  if (gridDim.x > 1) {
    // device-coherent hand-over to the row's last workgroup
    __hip_atomic_store(part + (int64_t)row * gridDim.x + blockIdx.x, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    last = __hip_atomic_fetch_add(counters + row * kDecodeCounterStride, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    if (!last) return;
    for (unsigned i = 0; i < gridDim.x; ++i) {
      const unsigned long long x = __hip_atomic_load(part + (int64_t)row * gridDim.x + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      mine = x < mine ? x : mine;
    }
  }
  a.next_index[row] = (int32_t)(mine & 0xffffffffull);
}

// ---- k > 1, a row over several workgroups -----------------------------------------------------
//
// A row has few keys for a device (8 rows of 16384 slots) and many for one workgroup: with one workgroup per row the
// choice of 1024 slots took 40 us, bound by one compute unit's LDS and instruction issue. Lists of 256, 512 or 1024 keys are
// sorted side by side instead, and ranks need no hand-over between workgroups but the launch boundary.
// List c of a row takes the 16-slot blocks c, c + C, c + 2C, ... (C lists): old and new tokens lie in runs of slots, and
// this way every list is a sample of the whole row, so that the bound below is tight whatever the order of the slots. Blocks of
// 64 slots were too long for that: 1024 new slots in a run met 16 lists of 64 (ranks of 1024 among 16 x 1024 slots 11.2 -> 6.4 us).

constexpr int LIST = 1024;  // slots a workgroup of the passes before the sort, one per thread
constexpr int RANK_THREADS = 512;
constexpr int RANK_STAGED = 6144;  // keys of the lists' heads that the ranking workgroup holds in LDS

// What the launches hand on, per (row, part) or (row, list).
struct SelectLists {
  unsigned long long* keys;  // sorted keys
  float* part_z;             // v_norm: sum of v_norm * w (nullptr: the statistics' workgroups add the row up themselves)
  float* stats;              // q_errors: extremes of the compared value and of the errors (4 floats)
  int C;                     // parts of LIST slots: norm and statistics
  int lists;                 // sorted lists
};
__device__ __forceinline__ int part_slot(int c, int C, int t) { return ((t >> 6) * C + c) * 64 + (t & 63); }
__device__ __forceinline__ int list_slot(int c, int lists, int t) { return ((t >> 4) * lists + c) * 16 + (t & 15); }

__global__ __launch_bounds__(LIST) void list_norm_kernel(const kvx_h2o_args a, const SelectLists sl) {
  __shared__ float red[LIST / 64];
  const int c = blockIdx.y, row = blockIdx.x, b = row / a.Hkv, hh = row % a.Hkv;
  const int slot = part_slot(c, sl.C, threadIdx.x);
  float x = 0.0f;
  if (slot < a.kv_len) x = a.v_norm[b * a.sc_stride_b + hh * a.sc_stride_h + slot] * a.w[(int64_t)row * a.kv_len + slot];
  x = block_reduce(x, red, [](float u, float v) { return u + v; });
  if (threadIdx.x == 0) sl.part_z[row * sl.C + c] = x;
}

__device__ __forceinline__ float wave_total(float x);

// Sum of v_norm * w over a row: of the parts' sums, or from the products by every workgroup of LIST threads for itself, the same bits
// (64 products, the 16 wavefronts of a part, the parts). Rows of at most Z_SLOTS slots are added up anew by each of their workgroups
// (24000 products a workgroup of 16 rows of 6000: norm and statistics 9.7 us as two launches, 7.9 as one); a launch of its own reads a long
// row once. Ahead of the sort the launch stays for all rows: workgroups of 256 threads took 9 us more for the sum.
constexpr int Z_SLOTS = 8192, Z_PARTS = Z_SLOTS / LIST;
template <int THREADS>
__device__ __forceinline__ float parts_norm(const SelectLists& sl, float* red, int row) {
  const float z = (int)threadIdx.x < sl.C ? sl.part_z[row * sl.C + threadIdx.x] : 0.0f;
  return block_reduce<THREADS>(z, red, [](float u, float v) { return u + v; });
}
__device__ __forceinline__ float row_norm(const kvx_h2o_args& a, int C, int row, int b, int hh) {
  constexpr int WAVES = LIST / 64;
  __shared__ float red[WAVES * Z_PARTS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float *vn = a.v_norm + b * a.sc_stride_b + hh * a.sc_stride_h, *w = a.w + (int64_t)row * a.kv_len;
  float x[Z_PARTS];
#pragma unroll
  for (int c = 0; c < Z_PARTS; ++c) {
    const int slot = part_slot(c, C, threadIdx.x);
    x[c] = c < C && slot < a.kv_len ? vn[slot] * w[slot] : 0.0f;
  }
#pragma unroll
  for (int c = 0; c < Z_PARTS; ++c) {
    const float t = wave_total(x[c]);
    if (lane == 0) red[wave * Z_PARTS + c] = t;
  }
  __syncthreads();
  float z = 0.0f;
  if (lane < C) {
    z = red[lane];
    for (int i = 1; i < WAVES; ++i) z += red[i * Z_PARTS + lane];
  }
  return wave_total(z);
}

// What a thread needs of its slot, asked for at once and ahead of the sums over the row, behind whose barriers each would be a latency of its own.
struct Slot {
  float score, w, v_norm;
  int position;
};
__device__ __forceinline__ Slot load_slot(const kvx_h2o_args& a, int row, int b, int hh, int slot) {
  const int64_t off = b * a.sc_stride_b + hh * a.sc_stride_h + slot;
  const bool in = slot < a.kv_len;
  Slot s;
  s.score = in ? a.scores[off] : 0.0f;
  s.w = in && a.w ? a.w[(int64_t)row * a.kv_len + slot] : 0.0f;
  s.v_norm = in && a.w && a.v_norm ? a.v_norm[off] : 0.0f;
  s.position = in && a.normalize ? a.token_pos[b * a.tp_stride_b + hh * a.tp_stride_h + slot] : 0;
  return s;
}
// The slot's score after the update (stored); `z`: the row's sum of v_norm * w. Every product and sum rounded on its own.
__device__ __forceinline__ float updated_score(const kvx_h2o_args& a, const Slot& s, float z, int b, int hh, int slot) {
  if (!a.w) return s.score;
  float inst = s.w;
  if (a.v_norm) inst = __fmul_rn(__fmul_rn(s.v_norm, s.w) / z, (float)a.q_len);
  const float v = __fadd_rn(s.score, inst);
  if (slot < a.kv_len) a.scores[b * a.sc_stride_b + hh * a.sc_stride_h + slot] = v;
  return v;
}

// q_errors: the update and the lists' extremes, before anything can be compared
__global__ __launch_bounds__(LIST) void list_stats_kernel(const kvx_h2o_args a, const SelectLists sl) {
  __shared__ float red[LIST / 64];
  const int c = blockIdx.y, row = blockIdx.x, b = row / a.Hkv, hh = row % a.Hkv;
  const int slot = part_slot(c, sl.C, threadIdx.x);
  const bool in = slot < a.limit;
  const float qe = in ? a.q_errors[b * a.sc_stride_b + hh * a.sc_stride_h + slot] : 0.0f;
  const Slot s = load_slot(a, row, b, hh, slot);
  const float z = !a.w || !a.v_norm ? 1.0f : sl.part_z ? parts_norm<LIST>(sl, red, row) : row_norm(a, sl.C, row, b, hh);
  const float v = updated_score(a, s, z, b, hh, slot);
  const float cv = in ? residency_of(v, a, s.position) : 0.0f;
  const f32x4_t ex = block_extremes<LIST>(f32x4_t{in ? cv : INFINITY, in ? cv : -INFINITY, in ? qe : INFINITY, in ? qe : -INFINITY});
  if (threadIdx.x == 0) *(f32x4_t*)(sl.stats + ((int64_t)row * sl.C + c) * 4) = ex;
}

// Sum over the wavefront in the order of block_reduce's exchanges.
__device__ __forceinline__ float wave_total(float x) {
  auto add = [](float v, uint32_t y) { return v + __uint_as_float(y); };
  x = add(x, lane_xor<32>(__float_as_uint(x)));
  x = add(x, lane_xor<16>(__float_as_uint(x)));
  x = add(x, lane_xor<8>(__float_as_uint(x)));
  x = add(x, lane_xor<4>(__float_as_uint(x)));
  x = add(x, lane_xor<2>(__float_as_uint(x)));
  return add(x, lane_xor<1>(__float_as_uint(x)));
}

template <int S>
__device__ __forceinline__ unsigned long long sort_step(unsigned long long x, int size) {
  const unsigned long long y = ((unsigned long long)lane_xor<S>((uint32_t)(x >> 32)) << 32) | lane_xor<S>((uint32_t)x);
  const bool keep_min = ((threadIdx.x & S) == 0) == ((threadIdx.x & size) == 0);
  return (y < x) == keep_min ? y : x;
}

// Bitonic sort of L keys, one a thread: steps between lanes of a wavefront on the vector ALU, the others through LDS (two
// buffers in turn: one barrier each).
template <int L>
__device__ __forceinline__ unsigned long long sort_list(unsigned long long x, unsigned long long (&buf)[2][L]) {
  const int t = threadIdx.x;
  int which = 0;
#pragma unroll 1
  for (int size = 2; size <= L; size <<= 1) {
#pragma unroll 1
    for (int stride = size >> 1; stride >= 64; stride >>= 1) {
      buf[which][t] = x;
      __syncthreads();
      const unsigned long long y = buf[which][t ^ stride];
      const bool keep_min = ((t & stride) == 0) == ((t & size) == 0);
      x = (y < x) == keep_min ? y : x;
      which ^= 1;
    }
    if (size >= 64) x = sort_step<32>(x, size);
    if (size >= 32) x = sort_step<16>(x, size);
    if (size >= 16) x = sort_step<8>(x, size);
    if (size >= 8) x = sort_step<4>(x, size);
    if (size >= 4) x = sort_step<2>(x, size);
    x = sort_step<1>(x, size);
  }
  return x;
}

template <int L>
__global__ __launch_bounds__(L, 8) void list_sort_kernel(const kvx_h2o_args a, const SelectLists sl) {
  __shared__ float red[L / 64];
  __shared__ unsigned long long buf[2][L];
  const int tid = threadIdx.x, c = blockIdx.y, row = blockIdx.x, b = row / a.Hkv, hh = row % a.Hkv;
  const int slot = list_slot(c, sl.lists, tid);
  const bool in = slot < a.limit;
  unsigned long long x = ~0ull;
  if (a.q_errors) {
    const int64_t off = b * a.sc_stride_b + hh * a.sc_stride_h;
    const float v = in ? a.scores[off + slot] : 0.0f, qe = in ? a.q_errors[off + slot] : 0.0f;
    const int position = in && a.normalize ? a.token_pos[b * a.tp_stride_b + hh * a.tp_stride_h + slot] : 0;
    float v4[4] = {INFINITY, -INFINITY, INFINITY, -INFINITY};
    const float* st = sl.stats + (int64_t)b * a.Hkv * sl.C * 4;
    for (int i = tid; i < a.Hkv * sl.C; i += L) {
      const f32x4_t s4 = *(const f32x4_t*)(st + i * 4);
      v4[0] = fminf(v4[0], s4[0]);
      v4[1] = fmaxf(v4[1], s4[1]);
      v4[2] = fminf(v4[2], s4[2]);
      v4[3] = fmaxf(v4[3], s4[3]);
    }
    const f32x4_t ex = block_extremes<L, (L > 512 ? 8 : L / 64)>(f32x4_t{v4[0], v4[1], v4[2], v4[3]});
    Modify m;
    m.smin = ex[0];
    m.sden = ex[1] - m.smin;
    m.qmin = ex[2];
    m.qden = ex[3] - m.qmin;
    m.c = (float)a.combination;
    m.c2 = (float)((a.combination - 1.0) / 2.0);
    m.c3 = (float)(1.0 - a.combination);
    if (in) x = ((unsigned long long)ordered_bits(combined_value(residency_of(v, a, position), qe, m)) << 32) | (unsigned)slot;
  } else {
    const Slot s = load_slot(a, row, b, hh, slot);
    const float z = a.w && a.v_norm ? parts_norm<L>(sl, red, row) : 1.0f;
    const float v = updated_score(a, s, z, b, hh, slot);
    if (in) x = ((unsigned long long)ordered_bits(residency_of(v, a, s.position)) << 32) | (unsigned)slot;
  }
  x = sort_list<L>(x, buf);
  if (sl.lists == 1) {  // the row is one list
    if (tid < a.k) a.next_index[(int64_t)row * a.k + tid] = (int32_t)(x & 0xffffffffull);
  } else {
    sl.keys[((int64_t)row * sl.lists + c) * L + tid] = x;
  }
}

// Ranks of the keys of list c. `per` = ceil(k / C) keys of every list are at or below U, the largest of the lists'
// per-th keys, so the first k keys of the row are all at or below U: about per of each list when the lists are alike.
// Only those are ranked: a key's rank is its place in its list plus its places in the others, found by binary search in
// the lists' heads (2^staged keys each, in LDS; in memory beyond them, a latency a step). The list with the most keys at or below U has
// about 2 per + 14 of them over many lists and rows, and one search beyond the heads is what the launch waits for: with heads of 2 per keys (16 at least),
// sort and ranks of 256 of 8192 slots, 12 rows, 14.9 us, now 10.8; 16 of 4096 slots, 64 rows, 13.6, now 11.7.
template <int L>
__global__ __launch_bounds__(RANK_THREADS) void list_rank_kernel(const unsigned long long* __restrict__ lists, int C, int k, int per, int staged, int32_t* __restrict__ next) {
  __shared__ unsigned long long head[RANK_STAGED];
  __shared__ uint32_t rank[L];
  __shared__ unsigned long long wmax[RANK_THREADS / 64];
  const int tid = threadIdx.x, c = blockIdx.y, row = blockIdx.x, S = 1 << staged;
  const unsigned long long* base = lists + (int64_t)row * C * L;
  for (int i = tid; i < C << staged; i += RANK_THREADS) head[i] = base[(i >> staged) * L + (i & (S - 1))];
  unsigned long long u = 0ull;
  for (int i = tid; i < C; i += RANK_THREADS) {
    const unsigned long long x = base[i * L + per - 1];
    u = x > u ? x : u;
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const unsigned long long o = __shfl_xor(u, off, 64);
    u = o > u ? o : u;
  }
  if ((tid & 63) == 0) wmax[tid >> 6] = u;
  for (int i = tid; i < L; i += RANK_THREADS) rank[i] = 0u;
  __syncthreads();
  for (int i = 0; i < RANK_THREADS / 64; ++i) u = wmax[i] > u ? wmax[i] : u;
  u = u == ~0ull ? u - 1 : u;  // places without a slot are never ranked
  // keys of `list` below x
  auto below = [&](int list, unsigned long long x) {
    const unsigned long long* h = head + (list << staged);
    int lo = 0;
    for (int half = S >> 1; half > 0; half >>= 1) lo += h[lo + half - 1] < x ? half : 0;
    lo += h[lo] < x ? 1 : 0;
    if (lo == S && S < L) {
      for (int n = L - S; n > 0;) {
        const int half = n >> 1;
        const bool up = base[list * L + lo + half] < x;
        lo += up ? half + 1 : 0;
        n = up ? n - half - 1 : half;
      }
    }
    return lo;
  };
  auto at = [&](int e) { return e < S ? head[(c << staged) + e] : base[c * L + e]; };
  const int n = below(c, u + 1);
  for (int i = tid; i < n * C; i += RANK_THREADS) {
    const int list = i / n, e = i - list * n;
    const int r = list == c ? e : below(list, at(e));
    if (r) atomicAdd(&rank[e], (uint32_t)r);
  }
  __syncthreads();
  for (int e = tid; e < n; e += RANK_THREADS)
    if (rank[e] < (uint32_t)k) next[(int64_t)row * k + rank[e]] = (int32_t)(at(e) & 0xffffffffull);
}

// ---- k > 1, one workgroup per row --------------------------------------------------------------

// CACHED: the row's ordered keys live in LDS after the first pass (rows of up to ~36K slots), so the
// radix passes and the gather never go back to global memory.
// Selections of more than MAX_PASS_K slots run as several launches: each takes the next a.k smallest
// (value, slot) keys above `bound` (the last key of the launch before, per row) and leaves its own last
// key there. out_off / out_stride place the launch's slots inside the row of next_index.
struct SelectPass {
  unsigned long long* bound;  // per row, or nullptr: a single launch
  int lower;                  // 1: only keys above bound[row] take part
  int out_off, out_stride;
};

template <bool CACHED>
__global__ __launch_bounds__(SEL_THREADS) void update_select_kernel(const kvx_h2o_args a, int kpad, const float* stats, const SelectPass ps) {
  extern __shared__ __align__(16) unsigned char dyn_lds[];
  unsigned long long* cand = (unsigned long long*)dyn_lds;    // kpad entries
  uint32_t* keys = (uint32_t*)(dyn_lds + (size_t)kpad * 8);   // a.limit entries (CACHED only)
  __shared__ uint32_t hist[256];
  __shared__ uint32_t wave_cnt[SEL_THREADS / 64];
  __shared__ uint32_t sh_prefix, sh_krem, sh_diff;
  __shared__ int sh_hi;

  const int tid = threadIdx.x;
  const int row = blockIdx.x;
  const int b = row / a.Hkv, hh = row % a.Hkv;
  float* sc = a.scores + b * a.sc_stride_b + hh * a.sc_stride_h;
  const float* w = a.w ? a.w + (int64_t)row * a.kv_len : nullptr;
  const int32_t* tpr = a.token_pos ? a.token_pos + b * a.tp_stride_b + hh * a.tp_stride_h : nullptr;
  const Modify md = load_modify(a, stats, b, hh);
  // keys at or below the bound were taken by an earlier launch: they get the largest key and so never
  // come before a key still to be taken
  const unsigned long long bound = ps.lower ? ps.bound[row] : 0ull;
  const uint32_t bound_u = (uint32_t)(bound >> 32), bound_i = (uint32_t)bound;
  auto live_key = [&](float v, int i) -> uint32_t {
    const uint32_t u = ordered_bits(select_value(v, a, tpr, i, md));
    if (ps.lower && (u < bound_u || (u == bound_u && (uint32_t)i <= bound_i))) return 0xffffffffu;
    return u;
  };

  // pass 0: scores += w (every later pass of this thread touches the slots it wrote here) and the keys
  // One workgroup walks the whole row: batches of 8 loads per array are issued before anything is
  // stored, otherwise the stores to sc (which may alias w for all the compiler knows) serialise the
  // loads and the pass costs one memory round trip per element of a thread.
  const int n0 = max(a.kv_len, a.limit);
  constexpr int PB = 8;
  for (int i0 = tid; i0 < n0; i0 += PB * SEL_THREADS) {
    float sv[PB], wv[PB];
#pragma unroll
    for (int j = 0; j < PB; ++j) {
      const int i = i0 + j * SEL_THREADS;
      sv[j] = i < n0 ? sc[i] : 0.0f;
      wv[j] = (w && i < a.kv_len) ? w[i] : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < PB; ++j) {
      const int i = i0 + j * SEL_THREADS;
      if (i >= n0) break;
      float v = sv[j];
      if (w && i < a.kv_len) {
        v += wv[j];
        sc[i] = v;
      }
      if (CACHED && i < a.limit) keys[i] = live_key(v, i);
    }
  }
  auto key_of = [&](int i) -> uint32_t {
    if constexpr (CACHED) return keys[i];
    else return live_key(sc[i], i);
  };

  for (int i = tid; i < kpad; i += SEL_THREADS) cand[i] = ~0ull;
  if (tid == 0) {
    sh_prefix = 0;
    sh_krem = (uint32_t)a.k;
    sh_diff = 0;
  }
  __syncthreads();

  // Bits that all keys of the row share need no pass, and skipping them matters: scores of one row
  // share their sign and most of their exponent, so a first digit taken from bit 31 down would send
  // nearly every key to the same few LDS counters (same-address atomics serialise).
  {
    const uint32_t key0 = key_of(0);
    uint32_t diff = 0;
    for (int i = tid; i < a.limit; i += SEL_THREADS) diff |= key_of(i) ^ key0;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) diff |= __shfl_xor(diff, off, 64);
    if ((tid & 63) == 0 && diff) atomicOr(&sh_diff, diff);
    __syncthreads();
    if (tid == 0) {
      const int top = sh_diff ? 32 - __clz(sh_diff) : 0;  // bits [0, top) differ somewhere
      sh_hi = top;
      sh_prefix = top >= 32 ? 0u : (key0 >> top) << top;
    }
    __syncthreads();
  }
  constexpr int RB = 8;
  // radix select over the remaining bits, 8 at a time from the top: after a pass sh_prefix holds the
  // bits [lo, 32) of the k-th smallest key and sh_krem its rank among the keys sharing them.
  for (int hi = sh_hi; hi > 0;) {
    const int lo = max(hi - 8, 0);
    if (tid < 256) hist[tid] = 0;
    __syncthreads();
    const uint32_t prefix = sh_prefix;
    const uint32_t himask = hi >= 32 ? 0u : (0xffffffffu << hi);
    const uint32_t dmask = (1u << (hi - lo)) - 1u;
    // keys are fetched eight at a time: a loop of one dependent LDS read per counter update would run at
    // the latency of that read
    for (int i0 = tid; i0 < a.limit; i0 += RB * SEL_THREADS) {
      uint32_t u[RB];
#pragma unroll
      for (int j = 0; j < RB; ++j) {
        const int i = i0 + j * SEL_THREADS;
        u[j] = i < a.limit ? key_of(i) : ~prefix;  // a key that cannot match the prefix
      }
#pragma unroll
      for (int j = 0; j < RB; ++j)
        if (i0 + j * SEL_THREADS < a.limit && (u[j] & himask) == prefix) atomicAdd(&hist[(u[j] >> lo) & dmask], 1u);
    }
    __syncthreads();
    if (tid < 64) {
      // the digit where the running count reaches the rank: 4 bins per lane, wavefront prefix sum
      const uint32_t krem = sh_krem;
      uint32_t h4[4], tot = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        h4[j] = hist[4 * tid + j];
        tot += h4[j];
      }
      uint32_t incl = tot;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o = __shfl_up(incl, off, 64);
        if (tid >= off) incl += o;
      }
      uint32_t cum = incl - tot;  // keys in the bins before this lane's
      if (cum < krem && incl >= krem) {
        int j = 0;
        for (; j < 3; ++j) {
          if (cum + h4[j] >= krem) break;
          cum += h4[j];
        }
        sh_prefix = prefix | ((uint32_t)(4 * tid + j) << lo);
        sh_krem = krem - cum;
      }
    }
    __syncthreads();
    hi = lo;
  }
  const uint32_t ustar = sh_prefix;   // k-th smallest value
  const uint32_t need_eq = sh_krem;   // how many slots equal to it are taken (lowest slots first)
  const uint32_t nless = (uint32_t)a.k - need_eq;

  // gather: slots below ustar, then slots equal to it by ascending slot. Every wavefront owns a
  // contiguous stretch of the row, so slot order is (wavefront, step, lane) order: one sweep counts
  // both kinds per wavefront, a prefix over the wavefronts gives each its places, a second sweep writes
  // them (no atomics, nothing a step has to wait for).
  const int lane = tid & 63, wave = tid >> 6;
  constexpr int NWV = SEL_THREADS / 64;
  __shared__ uint32_t wave_less[NWV];
  const int chunk = ((a.limit + NWV - 1) / NWV + 63) / 64 * 64;
  const int c_begin = wave * chunk, c_end = min(c_begin + chunk, a.limit);
  uint32_t my_less = 0, my_eq = 0;
  for (int i0 = c_begin; i0 < c_end; i0 += 64 * RB) {
    uint32_t u[RB];
#pragma unroll
    for (int j = 0; j < RB; ++j) {
      const int i = i0 + 64 * j + lane;
      u[j] = i < c_end ? key_of(i) : 0xffffffffu;
    }
#pragma unroll
    for (int j = 0; j < RB; ++j) {
      const bool in = i0 + 64 * j + lane < c_end;
      my_less += (uint32_t)__popcll(__ballot(in && u[j] < ustar));
      my_eq += (uint32_t)__popcll(__ballot(in && u[j] == ustar));
    }
  }
  if (lane == 0) {
    wave_less[wave] = my_less;
    wave_cnt[wave] = my_eq;
  }
  __syncthreads();
  uint32_t pos_less = 0, rank = 0;  // places taken by the wavefronts before this one
  for (int ww = 0; ww < wave; ++ww) {
    pos_less += wave_less[ww];
    rank += wave_cnt[ww];
  }
  const bool place_eq = rank < need_eq && my_eq;
  if (my_less || place_eq) {
    for (int i0 = c_begin; i0 < c_end; i0 += 64) {
      const int i = i0 + lane;
      const uint32_t u = i < c_end ? key_of(i) : 0xffffffffu;
      const bool less = i < c_end && u < ustar;
      const unsigned long long lm = __ballot(less);
      if (less) cand[pos_less + (uint32_t)__popcll(lm & ((1ull << lane) - 1ull))] = ((unsigned long long)u << 32) | (unsigned)i;
      pos_less += (uint32_t)__popcll(lm);
      if (place_eq) {
        const bool eq = i < c_end && u == ustar;
        const unsigned long long eqm = __ballot(eq);
        const uint32_t r = rank + (uint32_t)__popcll(eqm & ((1ull << lane) - 1ull));
        if (eq && r < need_eq) cand[nless + r] = ((unsigned long long)ustar << 32) | (unsigned)i;
        rank += (uint32_t)__popcll(eqm);
      }
    }
  }
  __syncthreads();

  // bitonic sort of kpad 64-bit keys. Comparator t of a stage with stride <= 64 only touches the 128
  // keys of its own wavefront's stretch, and a wavefront's LDS accesses execute in order: those
  // stages need no workgroup barrier.
  for (int size = 2; size <= kpad; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int t = tid; t < kpad / 2; t += SEL_THREADS) {
        const int lo = 2 * t - (t & (stride - 1));
        const int hi = lo + stride;
        const bool up = (lo & size) == 0;
        const unsigned long long x = cand[lo], y = cand[hi];
        if ((x > y) == up) {
          cand[lo] = y;
          cand[hi] = x;
        }
      }
      if (stride > 64 || (stride == 1 && 2 * size > 128)) __syncthreads();
      else __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    }
  __syncthreads();
  for (int j = tid; j < a.k; j += SEL_THREADS) a.next_index[(int64_t)row * ps.out_stride + ps.out_off + j] = (int32_t)(cand[j] & 0xffffffffull);
  if (ps.bound && tid == 0) ps.bound[row] = cand[a.k - 1];
}

}  // namespace

static bool is_variant(const kvx_h2o_args& a) { return a.v_norm != nullptr || a.q_errors != nullptr; }
constexpr int MAX_PASS_K = 4096;  // slots one launch of update_select_kernel sorts in LDS
// per row one 64-bit key: the running minimum of k == 1, or the bound handed from launch to launch when k > MAX_PASS_K
static size_t best_bytes(const kvx_h2o_args& a) {
  return (a.k == 1 || a.k > MAX_PASS_K) ? ((size_t)a.B * a.Hkv * sizeof(unsigned long long) + 15) / 16 * 16 : 0;
}

// what the one-workgroup-per-row form cannot do without
static size_t min_workspace(const kvx_h2o_args& a) { return best_bytes(a) + (a.q_errors ? (size_t)a.B * a.Hkv * 4 * sizeof(float) : 0); }

// Sorted lists for k > 1: taken while their number and size stay reasonable (256 parts of 1024 slots a row, 1 GiB), else
// (and where the caller's workspace does not hold them) one workgroup per row. Lists of 256 keys sort in 36 steps, 3 of them through LDS, of 512 in 45
// and 6, of 1024 in 55 and 10 by four times the wavefronts of a list of 256; but every candidate is looked up in all lists, by as many workgroups that
// each read the heads of all, and the shorter the lists, the more a run of new tokens fills one of them.
// So 256 while the device holds the workgroups side by side, three to a unit, and the look-ups are few for it; 512 up to 72 of them while the device holds their
// workgroups, three to a unit, and where neither those nor those of 1024 keys (half as many, two to a unit) fit at once and a row's look-ups are few; 1024 else. (The
// line was at 72 lists for any number of rows, priced against a sort of 1024 keys that had a unit to itself.)
// Whole choices in us, lists of 256, 512, 1024:
// 8 rows of 2336 slots 10.6, 9.1, 11.0; 32 x 3227 17.0, 15.1, 17.1; 16 x 30667 23.5, 20.0, 17.2; 32 x 27297 43.9, 33.9, 30.1; 64 x 14079 39.6, 30.7, 27.8;
// 64 x 34634 97.0, 66.9, 53.0; 4 x 38257 11.1, 10.2, 11.5; 8 x 45366 with errors 27.3, 20.7, 22.9; 402 of 49003, 4 rows: 512 14.8, 1024 13.7; of 512 and 1024, 526 of 27297, 32 rows 33.9, 30.1, 2 of 20422 33.9, 36.9,
// 558 of 26300, 16 rows 22.9, 18.5, 26 of 21229, 64 rows 34.3, 36.0.
// Rows of up to 1024 slots are one list whatever k is, the shortest that holds them: its sort ends the choice and hands nothing on (64 of 1000 slots, 32 rows: 9.9 us as
// four lists, 7.2 as one; in the 128 KiB of the static entry point, too little for four lists of 32 rows, 14.1 and 7.2); of 257 to 512 slots in a list of 512, not of 1024: 6.8 -> 5.0.
struct ListPlan {
  int C;         // parts of LIST slots per row, 0: not this way
  int L, lists;  // keys of a sorted list, lists per row
  size_t off_z, off_stats, total;
};
static ListPlan list_plan(const kvx_h2o_args& a) {
  ListPlan p{};
  if (a.k <= 1 || a.B <= 0 || a.Hkv <= 0 || a.kv_len <= 0 || (int64_t)a.B * a.Hkv > 65535) return p;  // (more rows: a workgroup each fills the device)
  const int64_t C = ((int64_t)a.kv_len + LIST - 1) / LIST, rows = (int64_t)a.B * a.Hkv;
  if (C > 256 || rows * C * LIST * 8 > (1ll << 30)) return p;
  p.C = (int)C;
  const int64_t n256 = (a.kv_len + 255) / 256, cus = num_cus();
  const bool few = C > 1 && a.kv_len <= 32768 && rows * n256 <= 3 * cus && a.k * n256 <= 32768 && rows * a.k * n256 <= 2048 * cus;
  const int64_t n512 = (a.kv_len + 511) / 512;
  const bool medium = C > 1 && n512 <= 72 && (rows * n512 <= 3 * cus || (rows * n512 > 4 * cus && a.k * n512 <= 3072));
  p.L = n256 == 1 || few ? 256 : n256 == 2 || medium ? 512 : LIST;
  p.lists = (a.kv_len + p.L - 1) / p.L;
  const size_t n = (size_t)(rows * C);
  p.off_z = p.lists > 1 ? (size_t)rows * p.lists * p.L * 8 : 0;
  p.off_stats = p.off_z + (n * 4 + 15) / 16 * 16;
  p.total = p.off_stats + n * 16;
  return p;
}

size_t h2o_workspace(const kvx_h2o_args& a) {
  const size_t least = min_workspace(a), lists = list_plan(a).total;
  return least > lists ? least : lists;
}

template <int L>
static void launch_sorted(const kvx_h2o_args& a, const SelectLists& sl, hipStream_t st) {
  const dim3 grid(a.B * a.Hkv, sl.lists);
  hipLaunchKernelGGL(list_sort_kernel<L>, grid, dim3(L), 0, st, a, sl);
  if (sl.lists == 1) return;
  const int per = (a.k + sl.lists - 1) / sl.lists;
  int staged = 4;
  while ((1 << staged) < 2 * per + 14 && (1 << staged) < L) ++staged;
  while (sl.lists << staged > RANK_STAGED) --staged;
  hipLaunchKernelGGL(list_rank_kernel<L>, grid, dim3(RANK_THREADS), 0, st, (const unsigned long long*)sl.keys, sl.lists, a.k, per, staged, a.next_index);
}

static int launch_lists(const kvx_h2o_args& a, const ListPlan& p, hipStream_t st) {
  SelectLists sl;
  char* ws = (char*)a.workspace;
  sl.keys = (unsigned long long*)ws;
  sl.part_z = a.kv_len > Z_SLOTS || !a.q_errors ? (float*)(ws + p.off_z) : nullptr;
  sl.stats = (float*)(ws + p.off_stats);
  sl.C = p.C;
  sl.lists = p.lists;
  // rows fastest: a row's workgroups, of every launch, are on the die (of eight, which take workgroups in turn) whose L2 the one before has written
  const dim3 grid(a.B * a.Hkv, p.C);
  if (a.w && a.v_norm && sl.part_z) hipLaunchKernelGGL(list_norm_kernel, grid, dim3(LIST), 0, st, a, sl);
  if (a.q_errors) hipLaunchKernelGGL(list_stats_kernel, grid, dim3(LIST), 0, st, a, sl);
  if (p.L == 256) launch_sorted<256>(a, sl, st);
  else if (p.L == 512) launch_sorted<512>(a, sl, st);
  else launch_sorted<LIST>(a, sl, st);
  KVX_HIP(hipGetLastError());
  return KVX_OK;
}

int launch_h2o_update_select(const kvx_h2o_args& a_in, hipStream_t st) {
  kvx_h2o_args a = a_in;
  const int rows = a.B * a.Hkv;
  if (rows == 0) return KVX_OK;
  KVX_REQUIRE(min_workspace(a) == 0 || (a.workspace && a.workspace_bytes >= min_workspace(a)), KVX_ERR_WORKSPACE,
              "kvx_h2o_update_select: workspace of %zu bytes needed", min_workspace(a));
  const ListPlan lists = list_plan(a);
  if (lists.C && a.workspace && a.workspace_bytes >= lists.total && ((uintptr_t)a.workspace & 15) == 0) return launch_lists(a, lists, st);
  float* stats = nullptr;
  if (is_variant(a)) {
    // the accumulation (and the batch statistics of the combination) first; what follows only selects
    if (a.q_errors) stats = (float*)((char*)a.workspace + best_bytes(a));
    if (a.w || stats) {
      hipLaunchKernelGGL(accumulate_kernel, dim3(rows), dim3(SEL_THREADS), 0, st, a, stats);
      KVX_HIP(hipGetLastError());
    }
    a.w = nullptr;
  }
  if (a.k == 1) {
    unsigned long long* best = (unsigned long long*)a.workspace;
    hipLaunchKernelGGL(argmin_init_kernel, dim3((rows + 255) / 256), dim3(256), 0, st, best, rows);
    KVX_HIP(hipGetLastError());
    hipLaunchKernelGGL(update_argmin_kernel, dim3((a.kv_len + 4095) / 4096, rows), dim3(256), 0, st, a, best, (const float*)stats);
    KVX_HIP(hipGetLastError());
    hipLaunchKernelGGL(argmin_finish_kernel, dim3((rows + 255) / 256), dim3(256), 0, st, best, a.next_index, rows);
    KVX_HIP(hipGetLastError());
    return KVX_OK;
  }
  // up to MAX_PASS_K slots per launch; a longer selection (the reference keeps the whole argsort when no chunk
  // size is set, keys_values/kvcache/attn_weights.py:773-774) continues above the last key of the launch before
  const int k_total = a.k;
  SelectPass ps;
  ps.bound = k_total > MAX_PASS_K ? (unsigned long long*)a.workspace : nullptr;
  ps.out_stride = k_total;
  for (int done = 0; done < k_total; done += MAX_PASS_K) {
    a.k = min(MAX_PASS_K, k_total - done);
    ps.lower = done > 0;
    ps.out_off = done;
    int kpad = 1;
    while (kpad < a.k) kpad <<= 1;
    // keys in LDS when the row fits beside the candidates (144 KB of the 160 KB of a compute unit)
    constexpr size_t kDynLimit = 144 * 1024;
    const size_t cached_bytes = (size_t)kpad * 8 + (size_t)a.limit * 4;
    if (cached_bytes <= kDynLimit) {
      if (cached_bytes > 48 * 1024)  // beyond the default dynamic LDS allowance (the setting is per device and kernel)
        KVX_HIP(hipFuncSetAttribute((const void*)update_select_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kDynLimit));
      hipLaunchKernelGGL(update_select_kernel<true>, dim3(rows), dim3(SEL_THREADS), cached_bytes, st, a, kpad, (const float*)stats, ps);
    } else {
      hipLaunchKernelGGL(update_select_kernel<false>, dim3(rows), dim3(SEL_THREADS), (size_t)kpad * 8, st, a, kpad, (const float*)stats, ps);
    }
    KVX_HIP(hipGetLastError());
    a.w = nullptr;  // the scores are updated once
  }
  return KVX_OK;
}

int launch_select_one(const kvx_h2o_args& a, const float* stats, int per_row, uint32_t* counters, unsigned long long* part, hipStream_t st) {
  const int wgs = (a.limit + SEL_ONE - 1) / SEL_ONE;
  hipLaunchKernelGGL(select_one_kernel, dim3(wgs, a.B * a.Hkv), dim3(SEL_THREADS), 0, st, a, stats, per_row, counters, part);
  KVX_HIP(hipGetLastError());
  return KVX_OK;
}
int select_one_parts(int limit) { return (limit + SEL_ONE - 1) / SEL_ONE; }

// ---- the same call for callers that cannot allocate -------------------------------------------
//
// The workspace of the selection (the per-row 64-bit minimum keys of k == 1, the per-row statistics of
// the Q-Hitter combination) lives in a file-scope device array instead of caller memory. `scratch`
// is only a host-side stand-in for that array: its device address is looked up once per device with
// hipGetSymbolAddress (every device holds its own copy at its own address) and only that address is
// handed to kernels.
constexpr size_t kStaticScratchBytes = 128 * 1024;
constexpr int kMaxDevices = 64;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

size_t h2o_static_scratch_bytes() { return kStaticScratchBytes; }

static int static_scratch_ptr(void** out) {
  static std::mutex mu;
  static void* ptrs[kMaxDevices] = {};
  int dev = 0;
  KVX_HIP(hipGetDevice(&dev));
  KVX_REQUIRE(dev >= 0 && dev < kMaxDevices, KVX_ERR_UNSUPPORTED, "kvx_h2o_update_select_static: device %d beyond the %d this library keeps scratch for", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(mu);
  if (!ptrs[dev]) {
    void* p = nullptr;
    KVX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    KVX_REQUIRE(p != nullptr, KVX_ERR_HIP, "kvx_h2o_update_select_static: no device address for the static scratch on device %d", dev);
    ptrs[dev] = p;
  }
  *out = ptrs[dev];
  return KVX_OK;
}

int launch_h2o_update_select_static(const kvx_h2o_args& a_in, hipStream_t st) {
  kvx_h2o_args a = a_in;
  const size_t need = min_workspace(a);
  KVX_REQUIRE(need <= kStaticScratchBytes, KVX_ERR_WORKSPACE,
              "kvx_h2o_update_select_static: B * Hkv = %d rows need %zu bytes of scratch, the static array holds %zu", a.B * a.Hkv, need,
              kStaticScratchBytes);
  void* p = nullptr;
  const int rc = static_scratch_ptr(&p);
  if (rc != KVX_OK) return rc;
  a.workspace = p;
  a.workspace_bytes = kStaticScratchBytes;
  return launch_h2o_update_select(a, st);
}

}  // namespace kvx
