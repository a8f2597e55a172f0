// Attention of chunks with few rows, or few keys, for gfx950: what sdpa_prefill.hip computes, in tiles of 16 or 32 (query, grouped
// head) rows of a KV head.
//
// The tiled kernel gives 32 rows to each of four (codes: eight) wavefronts and stages every tile of keys in LDS for all of them. With
// a handful of rows most of its wavefronts multiply zeros, over codes every tile is dequantised on the way with nobody to share it,
// and a short call is a serial chain: stage, barrier, scores, probabilities, barrier. Here the rows are the columns of both products
// and the wavefronts of a workgroup take the keys in turn, blocks of 32 straight from memory (key_blocks.h), two in flight each, without
// barriers in the loop; a block's operands are dequantised once and serve all the columns. The wavefronts' partial results meet in LDS
// at the end. Bound by the read of K and V, and where that is short by latency: loads, a few blocks, the exchange, the merge.
//
// Attention without weights, calls in a row, in the tiled kernel -> here: 20 rows over 32 x 36928 keys of 128, 8-bit codes 176 -> 87 us, 4-bit
// 176 -> 67; 8 over 8 x 8192, 8-bit 19.2 -> 11.8, plain 17.0 -> 10.4; 60 of 64 over 8 x 9000, 8-bit 19.5 -> 14.0; 64 of 256 over 4 x 10590, 8-bit
// 40.6 -> 28.3; 200 over 8 x 2000, 8-bit 25.3 -> 18.5, plain 21.4 -> 14.8; 512 over 8 x 600, 8-bit 22.1 -> 11.4, plain 17.5 -> 9.1; 512 of 64 over
// 8 x 1024, plain 14.5 -> 8.8.
//
// With weights, a call whose workgroups fit the device at once keeps the logits of each in LDS and ends there too (finish_weights, weights_plan):
// the second pass over Q K^T and its launch, half of such a call, go.
#include <float.h>

#include <atomic>
#include <chrono>
#include <random>

#include "key_blocks.h"
#include "prefill_params.h"

namespace kvx {
namespace {

constexpr int WAVES = 4;
constexpr float kNegBig = -FLT_MAX;  // running maximum before the first visible key: finite (no inf - inf), and below the logits of any key

// Two workgroups per compute unit where the accumulators (NC D / 4 registers) leave room for two blocks in flight, else one: with 32
// rows of 128 a bound of two spills the blocks of plain and 8-bit keys, 4-bit ones fit.
constexpr int per_cu(int D, int NC, bool u4) { return NC * D <= 128 || (NC * D == 256 && D == 128 && u4) ? 2 : 1; }

// Attention with weights in one launch (the template argument W): what a call needs beside PrefillParams.
struct RowsWeights {
  float* w;
  u32x4_t* sums;                    // [group][row block][pair of keys]: sums over the rows of a block, and the token (store_marked); NULL with one block
  u32x4_t* pairs;                   // [group][row block][row][split]: a split's maximum and sum, and the token (store_marked)
  unsigned long long* missed_rows;  // flags [group][row block][split]: a split whose wait for the others ran out
  unsigned long long* missed_sums;  // flags [group][split][row block]: a block whose wait for the others' sums ran out
  float* logits;                    // [group][row block][split][split_keys columns]: of splits whose wait ran out
  unsigned long long token;         // a number that no other call has
  int32_t split_keys;               // keys of a split, whole tiles
  int32_t spin_limit, poll_sleep;
  float inv_g;
};

// Values that cross workgroups inside one launch: device-coherent (they bypass the caches that the dies do not share).
template <typename P>
__device__ __forceinline__ auto coherent_load(P q) { return __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename P, typename T>
__device__ __forceinline__ void coherent_store(P q, T v) { __hip_atomic_store(q, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// Two words and a call's token in 16 bytes, one store and one load of a lane: a word and half of the token in each aligned 8 bytes, which the memory
// that the dies share performs whole, so that a word is never taken for another call's.
constexpr int kCoherent = 16;  // sc1
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t words_at(const void* base) { return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 0xffffffff, 0x00027000); }
__device__ __forceinline__ void store_marked(rsrc_t at, uint32_t i, float x, float y, unsigned long long token) {
  __builtin_amdgcn_raw_buffer_store_b128(u32x4_t{__float_as_uint(x), (uint32_t)token, __float_as_uint(y), (uint32_t)(token >> 32)}, at, i * 16u, 0, kCoherent);
}
__device__ __forceinline__ u32x4_t load_marked(rsrc_t at, uint32_t i) {
  asm volatile("" ::: "memory");  // others write what is read: every time anew
  return __builtin_amdgcn_raw_buffer_load_b128(at, i * 16u, 0, kCoherent);
}
__device__ __forceinline__ bool is_marked(u32x4_t v, unsigned long long token) { return v[1] == (uint32_t)token && v[3] == (uint32_t)(token >> 32); }
__device__ __forceinline__ unsigned long long join_words(uint32_t lo, uint32_t hi) { return ((unsigned long long)hi << 32) | lo; }

template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}

constexpr int kMaxSplits = 64;  // of a block of rows whose splits wait for each other

// What a workgroup does with weights once its wavefronts' partial results are in LDS (red, rml) beside its logits (lg).
//
// It publishes its rows' outputs, maxima and sums, waits for those of the block's other splits, takes an equal share of the block's outputs
// and turns its logits into weights; their sums over the block's rows go to the workspace, where it waits for those of the other blocks
// for an equal share of the split's keys, and adds them in the order of the rows. All of a call's workgroups fit the device at once
// (weights_plan). Nothing has to be cleared before the launch: what is waited for carries the call's token of 64 bits, a number that no other call has
// (what the workspace held before equals it in one of 2^64 cases). A call that is being captured will be repeated with its token: a launch that clears goes before it.
//
// Both waits are bounded, by a few times what the whole call takes (weights_plan). One that runs out, as when other work, a second such call among it, holds
// the places of the workgroups that are waited for, says so in a flag, set by an exchange, and looks once more; what is still missing is then done by those that come later: each looks at the flags of the others once its own results
// have reached the memory that the dies share, so of two at least one finds what the other left. Several may do the same work: they write the same bits.
template <int D, int NC, bool F16>
__device__ __forceinline__ void finish_weights(const PrefillParams& p, const RowsWeights& x, float* lg, float* red, const float* rml, const int group, const int mblk, const int split,
                                               const int k_begin, const int k_end) {
  constexpr int COLS = 16 * NC, DS = D + 4, NT = 64 * WAVES;
  constexpr int J = NT / COLS, PER = kMaxSplits / J;  // lanes that share a row's splits, splits of a lane
  __shared__ __align__(16) float row_top[COLS], row_inv[COLS], row_lse[COLS];
  __shared__ uint32_t answer[WAVES];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = group / p.Hkv, kvh = group % p.Hkv, S = p.num_splits, rows = min(COLS, p.R - mblk * COLS);
  const int64_t block = (int64_t)group * p.m_blocks + mblk;
  const rsrc_t pairs = words_at(x.pairs + block * COLS * S);
  float* part_o = p.part_o + block * S * COLS * D;
  float* wt = red;  // [row][split]: 2^(maximum of the split - maximum of the row), once the outputs there have been read
  auto out_row = [&](int r) {
    const int row = mblk * COLS + r, qi = row / p.G, g = row - qi * p.G;
    return p.o + b * p.o_sb + (int64_t)(kvh * p.G + g) * p.o_sh + (int64_t)qi * p.o_st;
  };
  auto put_lse = [&] {
    if (tid >= rows) return;
    const int row = mblk * COLS + tid, qi = row / p.G, g = row - qi * p.G;
    p.lse[((int64_t)b * p.q_len + qi) * p.Hq + kvh * p.G + g] = row_lse[tid];
  };
  auto row_max = [&](int r) {
    float M = rml[2 * r];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) M = fmaxf(M, rml[2 * (w * COLS + r)]);
    return M;
  };
  // what all wavefronts agree on, for the whole workgroup
  auto agree = [&](bool mine) {
    if (lane == 0) answer[wave] = mine;
    __syncthreads();
    static_assert(WAVES == 4, "the wavefronts' answers");
    const bool all = answer[0] && answer[1] && answer[2] && answer[3];
    __syncthreads();
    return all;
  };
  float M = 0.0f, l = 0.0f;
  if (tid < COLS) {
    M = row_max(tid);
#pragma unroll
    for (int w = 0; w < WAVES; ++w) l += rml[2 * (w * COLS + tid) + 1] * fast_exp2(rml[2 * (w * COLS + tid)] - M);
    if (M == kNegBig) {  // no visible key
      M = -INFINITY;
      l = 0.0f;
    }
    if (S == 1) {
      row_top[tid] = M == -INFINITY ? 0.0f : M;
      row_inv[tid] = l > 0.0f && tid < rows ? 1.0f / l : 0.0f;
      row_lse[tid] = M + fast_log2(l);
      put_lse();
    }
  }
  if (S == 1) __syncthreads();
#pragma unroll
  for (int it = 0; it < COLS * (D / 4) / NT; ++it) {
    const int idx = tid + NT * it, r = idx / (D / 4), d4 = idx % (D / 4) * 4;
    if (r >= rows) break;
    const float top = row_max(r);
    f32x4_t o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < WAVES; ++w) o += *(const f32x4_t*)&red[(w * COLS + r) * DS + d4] * fast_exp2(rml[2 * (w * COLS + r)] - top);
    if (S > 1) {
      unsigned long long* to = (unsigned long long*)(part_o + ((int64_t)split * COLS + r) * D + d4);
      coherent_store(to, join_words(__float_as_uint(o[0]), __float_as_uint(o[1])));
      coherent_store(to + 1, join_words(__float_as_uint(o[2]), __float_as_uint(o[3])));
    } else {
      const float inv = row_inv[r];
      *(u32x2_t*)(out_row(r) + d4) = u32x2_t{pack_pair<F16>(o[0] * inv, o[1] * inv), pack_pair<F16>(o[2] * inv, o[3] * inv)};
    }
  }

  // the rows' maxima and sums, and the splits' weights, from the pairs; all workgroups of the block form the same bits
  auto row_state = [&](int limit) {
    const int r = tid / J, j = tid % J;
    float ms[PER], ls[PER];
    bool ok = false;
    for (int spin = 0; spin < limit; ++spin) {
      bool all = true;
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int s = j + J * u;
        u32x4_t v = {0xff800000u, (uint32_t)x.token, 0u, (uint32_t)(x.token >> 32)};
        if (s < S) v = load_marked(pairs, (uint32_t)(r * S + s));
        all = all && is_marked(v, x.token);
        ms[u] = __uint_as_float(v[0]);
        ls[u] = __uint_as_float(v[2]);
      }
      ok = __all(all);
      if (ok) break;
      const int pause = min(x.poll_sleep, 1 + (spin >> 2));
      for (int z = 0; z < pause; ++z) __builtin_amdgcn_s_sleep(8);
    }
    if (ok) {
      float M = ms[0], l = 0.0f;
#pragma unroll
      for (int u = 1; u < PER; ++u) M = fmaxf(M, ms[u]);
#pragma unroll
      for (int off = 1; off < J; off <<= 1) M = fmaxf(M, __shfl_xor(M, off, 64));
      const float top = M == -INFINITY ? 0.0f : M;
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const float f = fast_exp2(ms[u] - top);
        l += ls[u] * f;
        if (j + J * u < S) wt[r * kMaxSplits + j + J * u] = f;
      }
#pragma unroll
      for (int off = 1; off < J; off <<= 1) l += __shfl_xor(l, off, 64);
      if (j == 0) {
        row_top[r] = top;
        row_inv[r] = l > 0.0f && r < rows ? 1.0f / l : 0.0f;
        row_lse[r] = top + fast_log2(l);
      }
    }
    return agree(ok);
  };
  // the block's sums for the keys of split sp from its logits in lg: four lanes a key, four rows of each 16 a lane
  auto weigh = [&](int k0, int k1) {
    const rsrc_t sums = words_at(x.sums + block * ((p.kv_len + 1) / 2));
    const int quarter = tid & 3, seen = p.tp ? k1 : min(k1, p.input_pos + (mblk * COLS + rows - 1) / p.G + 1);  // keys behind are seen by no row here
    f32x4_t top[NC], inv[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      top[c] = *(const f32x4_t*)&row_top[16 * c + 4 * quarter];
      inv[c] = *(const f32x4_t*)&row_inv[16 * c + 4 * quarter];
    }
    for (int pair = tid >> 3; k0 + 2 * pair < k1; pair += NT / 8) {
      const int key = k0 + 2 * pair + ((tid >> 2) & 1);
      float t = 0.0f;
      if (key < seen) {
        const int k = key - k0, at = ((k & ~3) + ((k + (k >> 2)) & 3)) * 16 + 4 * quarter;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const f32x4_t s = *(const f32x4_t*)&lg[c * x.split_keys * 16 + at];
#pragma unroll
          for (int i = 0; i < 4; ++i) t = fmaf(fast_exp2(fmaf(s[i], p.c, -top[c][i])), inv[c][i], t);
        }
      }
      t += dpp_move<0x4E>(t);  // quad_perm [2,3,0,1]
      t += dpp_move<0xB1>(t);  // quad_perm [1,0,3,2]
      if (x.sums) {
        const float odd = dpp_move<0x141>(t);  // row_half_mirror: the other key's
        if ((tid & 7) == 0) store_marked(sums, (uint32_t)(k0 / 2 + pair), t, odd, x.token);
      } else if (quarter == 0 && key < k1) {
        x.w[(int64_t)group * p.kv_len + key] = t * x.inv_g;
      }
    }
  };
  // The share of split sp in the block's outputs, in pairs of values: L lanes a pair, each up to eight splits in flight. Behind it, the
  // stores that came before have reached memory (they have once the first loads are waited for).
  auto merge_share = [&](int sp) {
    const int E = rows * (D / 2), share = (E + S - 1) / S, e1 = min(share * (sp + 1), E);
    const int ll = S <= 8 ? 0 : S <= 16 ? 1 : S <= 32 ? 2 : 3, L = 1 << ll, j = tid & (L - 1);
    int e = share * sp + (tid >> ll);
    if (e >= e1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    for (; e < e1; e += NT >> ll) {  // the lanes of a pair leave the loop together
      const int r = e / (D / 2), d = e % (D / 2) * 2;
      const unsigned long long* from = (const unsigned long long*)(part_o + (int64_t)r * D + d);
      unsigned long long y[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) y[u] = coherent_load(from + (int64_t)min(j + L * u, S - 1) * (COLS * D / 2));
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float f = j + L * u < S ? wt[r * kMaxSplits + j + L * u] : 0.0f;
        a0 += __uint_as_float((uint32_t)y[u]) * f;
        a1 += __uint_as_float((uint32_t)(y[u] >> 32)) * f;
      }
      for (int off = 1; off < L; off <<= 1) {
        a0 += __shfl_xor(a0, off, 64);
        a1 += __shfl_xor(a1, off, 64);
      }
      if (j == 0) *(uint32_t*)(out_row(r) + d) = pack_pair<F16>(a0 * row_inv[r], a1 * row_inv[r]);
    }
  };
  // The share of block mb in the sums over all blocks of rows for the keys of a split, in the order of the rows; false: not all were there.
  auto add_share = [&](int mb, int k0, int k1, int limit) {
    const int all_pairs = (k1 - k0 + 1) / 2, n = (all_pairs + p.m_blocks - 1) / p.m_blocks, first = mb * n, count = min(n, all_pairs - first);
    const int kv_pairs = (p.kv_len + 1) / 2;
    const rsrc_t from = words_at(x.sums + (int64_t)group * p.m_blocks * kv_pairs + k0 / 2 + first);
    f32x2_t* all = (f32x2_t*)lg;  // [block][pair of the share]
    bool ok = true;
    int spin = 0;
    for (int i = tid; i < count * p.m_blocks; i += NT) {
      const int blk = i / count;
      u32x4_t v;
      for (;;) {
        v = load_marked(from, (uint32_t)(blk * kv_pairs + (i - blk * count)));
        if (is_marked(v, x.token) || ++spin >= limit) break;
        const int pause = min(2 * x.poll_sleep, 1 + (spin >> 1));
        for (int z = 0; z < pause; ++z) __builtin_amdgcn_s_sleep(4);
      }
      ok = ok && is_marked(v, x.token);
      all[i] = f32x2_t{__uint_as_float(v[0]), __uint_as_float(v[2])};
    }
    if (!agree(__all(ok))) return false;
    for (int i = tid; i < 2 * count; i += NT) {
      float t = 0.0f;
      for (int blk = 0; blk < p.m_blocks; ++blk) t += lg[2 * blk * count + i];
      const int key = k0 + 2 * first + i;
      if (key < k1) x.w[(int64_t)group * p.kv_len + key] = t * x.inv_g;
    }
    __syncthreads();
    return true;
  };
  auto set_flag = [&](unsigned long long* flag) {
    if (tid == 0) {
      const unsigned long long old = __hip_atomic_exchange(flag, x.token, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("s_waitcnt vmcnt(0)" : : "v"(old) : "memory");
    }
    __syncthreads();
  };
  auto is_set = [&](const unsigned long long* flag) {  // for the whole workgroup: a flag may be set at any moment
    if (tid == 0) answer[0] = coherent_load(flag) == x.token;
    __syncthreads();
    const bool set = answer[0];
    __syncthreads();
    return set;
  };
  auto any_flag = [&](const unsigned long long* flags, int n) {
    bool any = false;
    for (int i = tid; i < n; i += NT) any = any || coherent_load(flags + i) == x.token;
    return any;  // of this thread
  };
  // what follows the logits of split sp in lg
  auto tail = [&](int sp) {
    const int k0 = sp * x.split_keys, k1 = min(k0 + x.split_keys, p.kv_len);
    if (sp == 0 && S > 1) put_lse();
    weigh(k0, k1);
    if (S > 1) merge_share(sp);
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (!x.sums) return;
    __syncthreads();
    unsigned long long* missed = x.missed_sums + ((int64_t)group * S + sp) * p.m_blocks;
    const bool any = any_flag(missed, p.m_blocks);
    if (!add_share(mblk, k0, k1, x.spin_limit)) {
      set_flag(missed + mblk);
      (void)add_share(mblk, k0, k1, 1);
    }
    if (agree(!__any(any))) return;
    for (int mb = 0; mb < p.m_blocks; ++mb)
      if (mb != mblk && is_set(missed + mb)) (void)add_share(mb, k0, k1, max(x.spin_limit, 1));
  };

  if (S > 1) {
    unsigned long long* missed = x.missed_rows + block * S;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid < COLS) store_marked(pairs, (uint32_t)(tid * S + split), M, l, x.token);
    if (!row_state(x.spin_limit)) {
      float* to = x.logits + (block * S + split) * x.split_keys * COLS;
      for (int i = tid; i < x.split_keys * COLS; i += NT) coherent_store(to + i, lg[i]);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      set_flag(missed + split);
      if (!row_state(1)) return;
    }
    const bool any = any_flag(missed, S);  // asked for here, where this split's own pairs have been found
    tail(split);
    if (agree(!__any(any))) return;
    for (int sp = 0; sp < S; ++sp) {
      if (sp == split || !is_set(missed + sp)) continue;
      const float* from = x.logits + (block * S + sp) * x.split_keys * COLS;
      for (int i = tid; i < x.split_keys * COLS; i += NT) lg[i] = coherent_load(from + i);
      __syncthreads();
      tail(sp);
      __syncthreads();
    }
  } else {
    tail(0);
  }
}

template <int D, int NC, int KV, bool W>
__global__ __launch_bounds__(64 * WAVES, per_cu(D, NC, kv_is_u4(KV) && !W)) void sdpa_rows_kernel(const PrefillParams p, const RowsWeights x) {
  using Blocks = KeyBlocks<D, KV, false>;
  constexpr bool F16 = kv_elem_f16(KV);
  constexpr int KJ = Blocks::KJ, DPL = Blocks::DPL, CH = Blocks::CH, COLS = 16 * NC;
  constexpr int DS = D + 4;  // floats of a row in LDS: rows start 4 banks apart
  __shared__ __align__(16) float red[WAVES][COLS][DS];
  __shared__ float rml[WAVES][COLS][2];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, kg = lane >> 4;
  // A KV head's rows and keys stay on one XCD; with weights the splits of a block of rows wait for each other and are neighbours.
  const int group = W ? blockIdx.y : blockIdx.x, mblk = W ? blockIdx.z : blockIdx.y, split = W ? blockIdx.x : blockIdx.z;
  const int b = group / p.Hkv, kvh = group % p.Hkv;
  // With weights: the logits, [c][key][16]. The four keys of a lane group change places with its number, so that the four groups write to different
  // banks.
  extern __shared__ __align__(16) float lg[];
  int lg_at[4];  // key 4 kg + r of a tile
#pragma unroll
  for (int r = 0; r < 4; ++r) lg_at[r] = (4 * kg + ((r + kg) & 3)) * 16 + m;

  // This lane's column of every tile: row, query, position. The query rows of one tile are in registers; more are read from LDS as
  // they are multiplied, in operand order (kept in registers too they made the two blocks in flight spill).
  constexpr bool Q_LDS = NC > 1;
  __shared__ u32x4_t q_sh[Q_LDS ? NC * KJ * 64 : 1];
  u32x4_t qb[Q_LDS ? 1 : KJ];
  int qpos[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int row = mblk * COLS + 16 * c + m, rowc = min(row, p.R - 1);
    const int qi = rowc / p.G, g = rowc - qi * p.G;
    qpos[c] = p.input_pos + qi;
    const uint16_t* q = p.q + b * p.q_sb + (int64_t)(kvh * p.G + g) * p.q_sh + (int64_t)qi * p.q_st;
    if constexpr (!Q_LDS) {
#pragma unroll
      for (int e = 0; e < KJ; ++e) qb[e] = row < p.R ? *(const u32x4_t*)(q + Blocks::kslice(e, kg)) : u32x4_t{0u, 0u, 0u, 0u};
    } else {
      for (int e = wave; e < KJ; e += WAVES) q_sh[(c * KJ + e) * 64 + lane] = row < p.R ? *(const u32x4_t*)(q + Blocks::kslice(e, kg)) : u32x4_t{0u, 0u, 0u, 0u};
    }
  }
  const int row_first = min(mblk * COLS, p.R - 1), row_last = min(mblk * COLS + COLS, p.R) - 1;
  const int qpos_min = p.input_pos + row_first / p.G, qpos_max = p.input_pos + row_last / p.G;
  const int k_begin = split * p.tiles_per_split * BN;
  int k_end = min(k_begin + p.tiles_per_split * BN, p.kv_len);
  if (!p.tp) k_end = min(k_end, qpos_max + 1);  // slots hold positions 0, 1, 2, ...: nobody here sees the ones behind
  const int32_t* tp = p.tp ? p.tp + b * p.tp_sb + kvh * p.tp_sh : nullptr;
  Blocks blocks;
  blocks.init(p.k, p.v, p.k_scale, p.k_zp, p.v_scale, p.v_zp, b * p.k_sb + kvh * p.k_sh, b * p.v_sb + kvh * p.v_sh, b * p.qs_sb + kvh * p.qs_sh, p.k_st, p.v_st, p.qs_vec,
              m, kg, k_end);

  f32x4_t acc[NC][DPL];
  float m_run[NC], l_run[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    m_run[c] = kNegBig;
    l_run[c] = 0.0f;
#pragma unroll
    for (int t = 0; t < DPL; ++t) acc[c][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  }

  struct Keys {
    typename Blocks::Rows r;
    int32_t pos[8];  // of keys chunk0 + 16 (j / 4) + 4 kg + j % 4
  };
  auto issue = [&](Keys& x, int chunk0) {
    blocks.issue(x.r, chunk0);
    if (tp) {
      if (p.tp_vec && chunk0 + CH <= k_end) {
#pragma unroll
        for (int gi = 0; gi < 2; ++gi) {
          const int4 t = *(const int4*)(tp + chunk0 + 16 * gi + 4 * kg);
          x.pos[4 * gi] = t.x; x.pos[4 * gi + 1] = t.y; x.pos[4 * gi + 2] = t.z; x.pos[4 * gi + 3] = t.w;
        }
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) x.pos[j] = tp[min(chunk0 + 16 * (j >> 2) + 4 * kg + (j & 3), k_end - 1)];
      }
    }
  };
  auto consume = [&](Keys& x, int chunk0, int lg_keys) {
    f32x4_t s[NC][2];
#pragma unroll
    for (int e = 0; e < KJ; ++e) {
      const u32x4_t k0 = Blocks::k_operand(x.r, 0, e), k1 = Blocks::k_operand(x.r, 1, e);
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
        const u32x4_t q = Q_LDS ? q_sh[(c * KJ + e) * 64 + lane] : qb[Q_LDS ? 0 : e];
        s[c][0] = mfma_16x16x32<F16>(k0, q, e == 0 ? zero : s[c][0]);
        s[c][1] = mfma_16x16x32<F16>(k1, q, e == 0 ? zero : s[c][1]);
      }
    }
    // positions that some row may not see, and keys past the end
    const bool ragged = chunk0 + CH > k_end;
    bool masked = ragged || (!tp && chunk0 + CH - 1 > qpos_min);
    if (tp) {
      int top = x.pos[0];
#pragma unroll
      for (int j = 1; j < 8; ++j) top = max(top, x.pos[j]);
      masked = masked || __any(top > qpos_min);
    }
    if (masked) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = chunk0 + 16 * (j >> 2) + 4 * kg + (j & 3);
        const int pos = key >= k_end ? INT_MAX : (tp ? x.pos[j] : key);
#pragma unroll
        for (int c = 0; c < NC; ++c)
          if (pos > qpos[c]) s[c][j >> 2][j & 3] = -INFINITY;
      }
    }
    // this lane: column m of every tile, keys chunk0 + 16 gi + 4 kg + i
    u32x4_t pb[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if constexpr (W) {
        float* dst = lg + (c * lg_keys + chunk0 - k_begin) * 16;
#pragma unroll
        for (int j = 0; j < 8; ++j) dst[lg_at[j & 3] + 256 * (j >> 2)] = s[c][j >> 2][j & 3];
      }
      float mx = s[c][0][0];
#pragma unroll
      for (int j = 1; j < 8; ++j) mx = fmaxf(mx, s[c][j >> 2][j & 3]);
      mx *= p.c;
      // The reference is the exact maximum, not one that lags behind: the largest probability is then 1 and loses nothing in 16 bits. Up
      // to 4 % of a call; the output's error against 64 bits is 3 to 11 % below the tiled kernel's (a reference 2^8 behind: 7 % above to 3 % below).
      if (__any(mx > m_run[c])) {
        mx = max_halves(max_row_pairs(mx));  // the column's maximum over the four lane groups
        const float mn = fmaxf(m_run[c], mx), al = fast_exp2(m_run[c] - mn);
        m_run[c] = mn;
        l_run[c] *= al;
#pragma unroll
        for (int t = 0; t < DPL; ++t) acc[c][t] *= al;
      }
      float pv[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        pv[j] = fast_exp2(fmaf(s[c][j >> 2][j & 3], p.c, -m_run[c]));
        l_run[c] += pv[j];
      }
      pb[c] = u32x4_t{pack_pair<F16>(pv[0], pv[1]), pack_pair<F16>(pv[2], pv[3]), pack_pair<F16>(pv[4], pv[5]), pack_pair<F16>(pv[6], pv[7])};
    }
#pragma unroll
    for (int t = 0; t < DPL; ++t) {
      const u32x4_t v = Blocks::v_operand(x.r, t);
#pragma unroll
      for (int c = 0; c < NC; ++c) acc[c][t] = mfma_16x16x32<F16>(v, pb[c], acc[c][t]);
    }
  };

  // Two blocks in flight per wavefront: the loads of block i + 1 are issued before block i is consumed.
  constexpr int STRIDE = CH * WAVES;
  int chunk = k_begin + wave * CH;
  const int nsteps = max((k_end - chunk + STRIDE - 1) / STRIDE, 0);
  Keys ka, kb;
  if (nsteps > 0) issue(ka, chunk);
  if constexpr (Q_LDS) __syncthreads();
  for (int i = 0; i + 1 < nsteps; i += 2) {
    issue(kb, chunk + STRIDE);
    __builtin_amdgcn_sched_barrier(0);
    consume(ka, chunk, x.split_keys);
    __builtin_amdgcn_sched_barrier(0);  // the loads below reuse the registers consumed above
    issue(ka, min(chunk + 2 * STRIDE, k_end - 1));
    __builtin_amdgcn_sched_barrier(0);
    consume(kb, chunk + STRIDE, x.split_keys);
    __builtin_amdgcn_sched_barrier(0);
    chunk += 2 * STRIDE;
  }
  if (nsteps & 1) consume(ka, chunk, x.split_keys);

  // ---- the wavefronts' partials meet in LDS: a lane's values of column m are runs of consecutive d -----------------------------
  constexpr int RUN = Blocks::U4 ? DPL / 2 : DPL;  // d = dmap(t, 4 kg + i), consecutive over RUN values of t
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const float l = sum_halves(l_run[c] + __shfl_xor(l_run[c], 16, 64));
    if (kg == 0) {
      rml[wave][16 * c + m][0] = m_run[c];
      rml[wave][16 * c + m][1] = l;
    }
    float* row = red[wave][16 * c + m];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < DPL; t += RUN >= 4 ? 4 : 2) {
        float* d = row + Blocks::dmap(t, 4 * kg + i);
        if constexpr (RUN >= 4) *(f32x4_t*)d = f32x4_t{acc[c][t][i], acc[c][t + 1][i], acc[c][t + 2][i], acc[c][t + 3][i]};
        else *(f32x2_t*)d = f32x2_t{acc[c][t][i], acc[c][t + 1][i]};
      }
  }
  __syncthreads();
  if constexpr (W) {
    finish_weights<D, NC, F16>(p, x, lg, &red[0][0][0], &rml[0][0][0], group, mblk, split, k_begin, k_end);
    return;
  }
  const int64_t prow0 = ((int64_t)split * p.B * p.Hkv + group) * p.R;
#pragma unroll
  for (int it = 0; it < COLS * (D / 4) / (64 * WAVES); ++it) {
    const int idx = tid + 64 * WAVES * it, r = idx / (D / 4), d4 = idx % (D / 4) * 4;
    const int row = mblk * COLS + r;
    if (row >= p.R) break;
    float M = rml[0][r][0], l = 0.0f;
#pragma unroll
    for (int w = 1; w < WAVES; ++w) M = fmaxf(M, rml[w][r][0]);
    f32x4_t o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float sc = fast_exp2(rml[w][r][0] - M);
      l += rml[w][r][1] * sc;
      o += *(const f32x4_t*)&red[w][r][d4] * sc;
    }
    if (M == kNegBig) M = -INFINITY;  // no visible key
    if (p.num_splits == 1) {
      const float inv = l > 0.0f ? 1.0f / l : 0.0f;
      const int qi = row / p.G, g = row - qi * p.G;
      *(u32x2_t*)(p.o + b * p.o_sb + (int64_t)(kvh * p.G + g) * p.o_sh + (int64_t)qi * p.o_st + d4) =
          u32x2_t{pack_pair<F16>(o[0] * inv, o[1] * inv), pack_pair<F16>(o[2] * inv, o[3] * inv)};
      if (p.lse && d4 == 0) p.lse[((int64_t)b * p.q_len + qi) * p.Hq + kvh * p.G + g] = M + fast_log2(l);
    } else {
      *(f32x4_t*)(p.part_o + (prow0 + row) * D + d4) = o;
      if (d4 == 0) *(f32x2_t*)(p.part_ml + (prow0 + row) * 2) = f32x2_t{M, l};
    }
  }
}

// LDS of a workgroup beside its logits
constexpr int rows_lds(int D, int columns) {
  return WAVES * columns * (D + 4) * 4 + WAVES * columns * 8 + (columns > 16 ? columns * D * 2 : 0) + columns * 12 + 64;
}
constexpr int kLds = 160 * 1024;  // of a compute unit

template <int D, int NC, bool W>
int launch_dn(const PrefillParams& p, const RowsWeights& x, int kv, hipStream_t st) {
  const dim3 grid = W ? dim3(p.num_splits, p.B * p.Hkv, p.m_blocks) : dim3(p.B * p.Hkv, p.m_blocks, p.num_splits), block(64 * WAVES);
  const unsigned lds = W ? (unsigned)(x.split_keys * 16 * NC * 4) : 0;
#define KVX_ROWS_CASE(KV) \
  case KV: hipLaunchKernelGGL((sdpa_rows_kernel<D, NC, KV, W>), grid, block, lds, st, p, x); break;
  switch (kv) {
    KVX_ROWS_CASE(KVX_KV_U8)
    KVX_ROWS_CASE(KVX_KV_U4)
    KVX_ROWS_CASE(KVX_KV_U8_F16)
    KVX_ROWS_CASE(KVX_KV_U4_F16)
    default:
      if constexpr (D <= 128) {
        if (kv == KVX_KV_F16) hipLaunchKernelGGL((sdpa_rows_kernel<D, NC, KVX_KV_F16, W>), grid, block, lds, st, p, x);
        else hipLaunchKernelGGL((sdpa_rows_kernel<D, NC, KVX_KV_BF16, W>), grid, block, lds, st, p, x);
      }
  }
#undef KVX_ROWS_CASE
  KVX_HIP(hipGetLastError());
  return KVX_OK;
}
template <bool W>
int launch_columns(const PrefillParams& p, const RowsWeights& x, int D, int kv, hipStream_t st) {
  if (D == 64) return p.columns == 16 ? launch_dn<64, 1, W>(p, x, kv, st) : launch_dn<64, 2, W>(p, x, kv, st);
  if (D == 128) return p.columns == 16 ? launch_dn<128, 1, W>(p, x, kv, st) : launch_dn<128, 2, W>(p, x, kv, st);
  if constexpr (!W) {
    if (p.columns == 32) return launch_dn<256, 2, W>(p, x, kv, st);
  }
  return launch_dn<256, 1, W>(p, x, kv, st);
}

uint64_t mixed(uint64_t z) {  // splitmix64
  z += 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}
// A number that no other call has, and not zero.
uint64_t call_token() {
  static std::atomic<uint64_t> calls{0};
  static const uint64_t seed = [] {
    uint64_t s = mixed((uint64_t)(uintptr_t)&calls) ^ (uint64_t)std::chrono::steady_clock::now().time_since_epoch().count();
    try {
      std::random_device d;
      s ^= ((uint64_t)d() << 32) | d();
    } catch (...) {  // no source of random numbers: the address and the time
    }
    return s;
  }();
  const uint64_t t = mixed(seed + calls.fetch_add(1, std::memory_order_relaxed));
  return t ? t : 1;
}

}  // namespace

namespace {

// What a step of 128 keys (32 a wavefront) and the begin and end of a workgroup take, ns
int64_t step_ns(int D, bool plain, int columns) {
  int64_t ns = D == 64 ? 900 : D == 128 ? 1300 : 2600;
  if (plain) ns = ns * 77 / 100;
  return columns == 32 ? ns * (D == 64 ? 135 : 150) / 100 : ns;
}
int64_t ends_ns(int D, int columns) { return (columns == 16 ? 1000 : 2000) * D / 128; }

// Splits of the keys for workgroups of `columns` rows. Every workgroup walks its share at the same pace, so the walk ends with the
// most loaded compute unit: its rounds of 128 keys, and a second workgroup beside the first costs nine tenths of one more (it hides
// latency only, the pipes are shared). A workgroup's begin and end (first loads; the exchange in LDS) take a microsecond at 16 rows of 128, two at
// 32. The splits' merge is a launch, a chain over its splits (32 are one pass) and a read of their partials; combined in a score-sum launch that
// is there anyway they cost next to nothing, and one step a split is often the best (attention with weights of 8 rows over 4 x 3060 8-bit keys 14.6 us
// in 12 splits, 12.6 in 24; 32 over 4 x 384 plain keys 13.1 in one, 11.7 in 3). The rates are
// fits to calls of 2 to 1200 rows over 64 to 12000 keys: over codes a round takes 1.3 us at 16 rows of 128 (64: 0.9), half as much
// again at 32; the splits chosen take 1.0 % longer than the best of each call in the mean, without the workgroups' begin and end and
// with twice as much for a split 2.0 %. 200 rows over 8 x 2000 4-bit keys take 16.9 us in 4
// splits, 23.1 in 2, 20.6 in 5, 19.4 in 8 and 26.6 in 16; 17 as chosen.
RowsPlan plan_of(const kvx_sdpa_args& a, int columns, bool combined) {
  const bool plain = kv_is_plain(a.kv_dtype);
  const int per_unit = per_cu(a.D, columns / 16, kv_is_u4(a.kv_dtype));
  const int64_t rows = (int64_t)a.q_len * (a.Hq / a.Hkv), cus = num_cus();
  const int64_t wgs = (int64_t)a.B * a.Hkv * ((rows + columns - 1) / columns), steps = (a.kv_len + 127) / 128;  // 32 keys a wavefront
  const int64_t step = step_ns(a.D, plain, columns), ends = ends_ns(a.D, columns);
  RowsPlan best = {0, 0, INT64_MAX};
  int64_t best_per = 0;
  for (int64_t n = 1; n <= min(steps, (int64_t)64); ++n) {
    const int64_t per = (steps + n - 1) / n;
    if ((steps + per - 1) / per != n) continue;
    const int64_t c = (wgs * n + cus - 1) / cus;
    const int64_t walk = (per * step + ends) * (per_unit == 2 ? 180 * (c / 2) + 100 * (c % 2) : 100 * c) / 100;
    const int64_t merge = n == 1 ? 0 : (combined ? 300 + 30 * n : 2000 + 60 * n + (n > 32 ? 1000 : 0)) + n * a.B * a.Hq * a.q_len * (a.D * 4 + 8) / 4000;
    if (walk + merge < best.ns) {
      best = {columns, (int)n, walk + merge};
      best_per = per;
    }
  }
  // many short workgroups, fewer over a tile of keys: the tiled kernel (rows_plan)
  const int64_t all = wgs * best.splits;
  if (all > per_unit * cus && best_per <= (plain ? 3 : a.D == 256 ? 4 : 2)) return {0, 0, INT64_MAX};
  if (a.kv_len <= BN && a.D <= 128 && all * (columns / 16) > cus) return {0, 0, INT64_MAX};
  best.splits = (int)(((a.kv_len + BN - 1) / BN + 2 * best_per - 1) / (2 * best_per));  // splits of whole steps, in tiles
  return best;
}

}  // namespace

// The line between this kernel and the tiled one lies at the work a compute unit gets, in tiles of 32 rows by 128 keys: here every tile of
// rows reads (and over codes dequantises) the keys again, there 128 or 256 rows share them. Both sides, tiled -> here:
//   plain, 128     5 a unit  128 rows 27.5 -> 26.4, 512 rows (4) 37.4 -> 31.9;        6: 300 rows .98, 8: 600 rows .96 of the pace
//   plain, 64      8 a unit  512 rows 22.4 -> 22.3, 1000 rows 27.6 -> 27.0
//   codes, 128     6 a unit  300 rows 39.2 -> 37.8 (4-bit: 35.2), 512 rows (4) 41.1 -> 36.5;  7: 600 rows .88, 12: 96 rows .95
//   codes, 64      8-bit 10 a unit, 4-bit 7: 1000 rows (8) 33.8 -> 30.3, 300 rows (8) 31.1 -> 29.1;  4-bit 512 rows (7.5) .98
// At most 16 plain rows win while the keys stay in the last-level cache, 128 Ki of them (8 x 8192 20.3 -> 16.1, 32 x 36928 .98); at
// most 64 rows over codes always (64 over 8 x 30000 65 -> 62, 64 of 64 over 8 x 60000 65 -> 51). Rows of 256: the accumulators of plain
// keys' pipeline do not fit, over codes the tiled kernel is so slow that up to 128 rows win (128 over 4 x 15000 64 -> 50); above, a long call
// goes over a copy of the store in 16-bit rows.
// Many short workgroups stay there too (plan_of): one begins and ends with more than a step's work, so
// where the device takes the workgroups in turns and each has up to three steps of 128 keys (over codes two, of 256 four) the tiled
// kernel's few win: 133 rows over 256 x 64 plain keys of 128 9.4 there, 25.5 here; 279 over 64 x 254 12.2, 22.7; 198 over 64 x 219 12.1, 15.8;
// 312 over 64 x 121 8-bit keys 13.8, 19.2; 66 of 256 over 128 x 512 8-bit keys 47.8, 53.8; but with four steps both take the same, and over codes three win by
// 1.1 to 2.2 here. Over at most a tile of keys more workgroups than units are too many, half of that at 32 rows: 35 over
// 128 x 64 5.2, 6.2.
RowsPlan rows_plan(const kvx_sdpa_args& a, bool combined) {
  const RowsPlan none = {0, 0, 0};
  const bool plain = kv_is_plain(a.kv_dtype);
  const int64_t rows = (int64_t)a.q_len * (a.Hq / a.Hkv), keys = (int64_t)a.B * a.Hkv * a.kv_len, es = plain ? 2 : 1;
  if ((int64_t)a.kv_len * a.k_stride_t * es >= (1ll << 32) || (int64_t)a.kv_len * a.v_stride_t * es >= (1ll << 32)) return none;
  const int64_t work = (rows + 31) / 32 * a.B * a.Hkv * ((a.kv_len + 127) / 128);  // 32 rows by 128 keys
  if (plain) {
    if (a.D == 256 || !((rows <= 16 && keys <= 128 * 1024) || work <= (a.D == 64 ? 8 : 5) * num_cus())) return none;
  } else {
    if ((a.D == 256 && rows > 128) || (rows > 64 && work > (a.D == 64 ? (kv_is_u4(a.kv_dtype) ? 7 : 10) : a.D == 128 ? 6 : 8) * num_cus())) return none;
  }
  const RowsPlan one = plan_of(a, 16, combined);
  if (rows <= 16) return one;
  const RowsPlan two = plan_of(a, 32, combined);
  return one.ns < two.ns ? one : two;
}

int launch_sdpa_rows(const PrefillParams& p, int D, int kv, hipStream_t st) { return launch_columns<false>(p, RowsWeights{}, D, kv, st); }

namespace {

// Attention with weights in one launch: rows of a workgroup and keys of a split with the least estimated time, 0 where a call takes two
// (two_launches_win among them).
//
// All workgroups have to fit the device at once, because they wait for each other: for the splits of their rows, and for the sums of the other
// blocks of rows. The waits take 2.5 us and 30 ns a split, a step half as long again as without weights, one of 64 keys six tenths of that; 172 of 220
// calls of 8 to 4000 rows over 100 to 65536 keys fit, and the plans chosen take 0.6 % longer than the best of 24 in the mean. Two launches ->
// one, calls in a row, us (about 10 of each are the host's): 512 rows over 2 x 1024 keys of 64 15.2 -> 11.6, over 2 x 512 14.5 -> 10.6, 1024 over 2 x 512
// 21.1 -> 10.9; of 128, 1024 over 2 x 1024 27.3 -> 17.8, 700 over 4 x 512 21.9 -> 14.4, 48 over 4 x 850 4-bit keys 13.4 -> 10.3, 36 over 8 x 4865 8-bit keys
// 22.1 -> 19.6; 256 of 256 over 2 x 1500 8-bit keys 33.9 -> 19.7. Splits of more than 11 steps (of 256: 8) are bound by the walk, and
// two launches share it out better: 322 rows over 2 x 12513 keys of 64 29.5 -> 35.7, 60 over 8 x 15028 30.4 -> 33.6, 210 of 256 over 16 x 1414
// 8-bit keys 50.7 -> 52.9.
//
// A wait is given up behind as many polls as take about ten times the estimate and 60 us more, the fetch of instructions by a first call among them; a poll
// is 1.5 to 2 us. What is given up is done by others from the workspace, for some us; held on to, the places of waiting workgroups are missing to those that they wait
// for, as between two calls on two streams that fill the device each.
struct WeightsPlan {
  int columns, splits, split_keys, polls;
};

// Whether two launches are estimated to take less than the one: for calls of several blocks of rows and several splits, where both waits are paid. (One split or
// rows of 256 values never lost in 378 calls, one block of rows 4 % at most; they are not priced.) Both prices are fits to GPU times of 1513 such calls of 17 to 2000 rows over 64 to 40000
// keys, 4 % off in the mean square. Always one launch took 2.3 % longer than the better of both in the mean (at most 23 %), two launches 7.1 % (53 %), as
// chosen 0.6 % (17 %). one / two launches, us: 105 rows over 16 x 756 15.7 / 14.8, 184 of 64 over 4 x 3428 8-bit keys 16.0 / 14.6, 20 of 64 over 2 x 15221
// 13.4 / 10.9, 120 over 8 x 1326 4-bit 19.3 / 16.1; 508 of 64 over 2 x 2336 14.1 / 17.1.
bool two_launches_win(const kvx_sdpa_args& a, const WeightsPlan& pl, int64_t one_ns) {
  const int64_t groups = (int64_t)a.B * a.Hkv, rows = (int64_t)a.q_len * (a.Hq / a.Hkv), blocks = (rows + 31) / 32, row_blocks = (rows + pl.columns - 1) / pl.columns;
  const int64_t c = (groups * row_blocks * pl.splits + num_cus() - 1) / num_cus();
  const bool narrow = a.D == 64;
  const int64_t one = one_ns * 115 / 100 + 5700 + (narrow ? 20 : 45) * row_blocks - 900 * (c - 1) - (narrow ? pl.split_keys * 3 / 2 : 0);
  int64_t second;  // and what both launches have besides their walks
  switch (score_sum_kind(a)) {
    case KVX_SCORE_SUM_SHORT: second = (narrow ? 6300 : 7000) + (narrow ? 1200 : 1300) * ((blocks + 3) / 4); break;
    case KVX_SCORE_SUM_STREAMED: {
      const int64_t rounds = (groups * ((a.kv_len + 63) / 64) + 2047) / 2048;
      second = narrow ? 6000 + 600 * rounds + 900 * blocks : 3200 + 1600 * rounds + 3200 * blocks;
      break;
    }
    default: second = 8200 + (narrow ? 230 : 400) * ((groups * ((a.kv_len + 255) / 256) + 255) / 256) * ((rows + 63) / 64);
  }
  if (!kv_is_plain(a.kv_dtype) && !narrow) second += 400;
  return one > second && one > second + prefill_ns(a) * (narrow ? 119 : 131) / 100;
}

WeightsPlan weights_plan(const kvx_sdpa_args& a) {
  WeightsPlan best = {0, 0, 0, 0};
  const bool plain = kv_is_plain(a.kv_dtype);
  const int64_t es = plain ? 2 : 1, cus = num_cus(), groups = (int64_t)a.B * a.Hkv, rows = (int64_t)a.q_len * (a.Hq / a.Hkv);
  if (a.num_splits > 1 || (plain && a.D == 256) || (a.D != 64 && a.D != 128 && a.D != 256)) return best;
  if ((int64_t)a.kv_len * a.k_stride_t * es >= (1ll << 32) || (int64_t)a.kv_len * a.v_stride_t * es >= (1ll << 32)) return best;
  const int64_t tiles = (a.kv_len + BN - 1) / BN;
  int64_t best_ns = INT64_MAX;
  for (int columns = 16; columns <= (rows > 16 && a.D < 256 ? 32 : 16); columns += 16) {
    const int64_t blocks = groups * ((rows + columns - 1) / columns), step = step_ns(a.D, plain, columns), ends = ends_ns(a.D, columns);
    for (int64_t n = 1; n <= min(tiles, (int64_t)(a.num_splits == 1 ? 1 : kMaxSplits)) && blocks * n <= 2 * cus; ++n) {
      const int64_t per = (tiles + n - 1) / n;
      if ((tiles + per - 1) / per != n || per > (a.D == 256 ? 16 : 22)) continue;
      const int64_t lds = rows_lds(a.D, columns) + per * BN * columns * 4;
      const int64_t per_unit = min((int64_t)per_cu(a.D, columns / 16, false), kLds / lds), c = (blocks * n + cus - 1) / cus;
      if (c > per_unit) continue;
      const int64_t walk = ((per / 2) * 15 + (per % 2) * 9) * step / 10 + ends;
      const int64_t ns = (c == 1 ? 100 : 180) * walk / 100 + (n > 1 ? 2500 + 30 * n : 0);
      if (ns < best_ns) {
        best_ns = ns;
        best = {columns, (int)n, (int)per * BN, (int)(40 + ns / 150)};
      }
    }
  }
  if (best.splits > 1 && rows > best.columns && a.D <= 128 && two_launches_win(a, best, best_ns)) return {0, 0, 0, 0};
  return best;
}

struct WeightsLayout {
  size_t pairs, sums, missed_rows, missed_sums, cleared, part_o, logits, total;  // cleared: bytes that a repeated call has to find without its token
};
WeightsLayout weights_layout(const kvx_sdpa_args& a, const WeightsPlan& pl) {
  const size_t groups = (size_t)a.B * a.Hkv, rows = (size_t)a.q_len * (a.Hq / a.Hkv), blocks = groups * ((rows + pl.columns - 1) / pl.columns), S = pl.splits;
  const bool split = S > 1, several = blocks > groups;
  WeightsLayout l;
  size_t off = 0;
  auto take = [&off](size_t bytes) {
    const size_t at = off;
    off += (bytes + 15) & ~(size_t)15;
    return at;
  };
  l.pairs = take(split ? blocks * S * pl.columns * 16 : 0);
  l.sums = take(several ? blocks * (((size_t)a.kv_len + 1) / 2) * 16 : 0);
  l.missed_rows = take(split ? blocks * S * 8 : 0);
  l.missed_sums = take(several ? blocks * S * 8 : 0);
  l.cleared = off;
  l.part_o = take(split ? blocks * S * pl.columns * a.D * 4 : 0);
  l.logits = take(split ? blocks * S * pl.columns * pl.split_keys * 4 : 0);
  l.total = off;
  return l;
}
__global__ void clear_kernel(u32x4_t* at, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) at[i] = u32x4_t{0u, 0u, 0u, 0u};
}
}  // namespace

size_t rows_weights_workspace(const kvx_sdpa_args& a) {
  const WeightsPlan pl = weights_plan(a);
  return pl.columns ? weights_layout(a, pl).total : 0;
}

bool rows_weights_plan(const kvx_sdpa_args& a, kvx_prefill_plan& plan) {
  const WeightsPlan pl = weights_plan(a);
  if (!pl.columns) return false;
  plan.one_launch = 1;
  plan.block_rows = pl.columns;
  plan.row_blocks = (a.q_len * (a.Hq / a.Hkv) + pl.columns - 1) / pl.columns;
  plan.splits = pl.splits;
  plan.split_keys = pl.split_keys;
  plan.polls = pl.polls;
  plan.teams = 1;
  return true;
}

int launch_rows_weights(const kvx_sdpa_args& a, hipStream_t st, bool& done) {
  done = false;
  const WeightsPlan pl = weights_plan(a);
  if (!pl.columns) return KVX_OK;
  const WeightsLayout l = weights_layout(a, pl);
  if (l.total && (!a.workspace || a.workspace_bytes < l.total)) return KVX_OK;
  PrefillParams p;
  common_params(p, a);
  p.columns = pl.columns;
  p.m_blocks = (p.R + pl.columns - 1) / pl.columns;
  p.num_splits = pl.splits;
  p.tiles_per_split = pl.split_keys / BN;
  char* ws = (char*)a.workspace;
  p.part_o = (float*)(ws + l.part_o);
  RowsWeights x{};
  x.w = a.w;
  x.inv_g = 1.0f / (float)p.G;
  x.sums = p.m_blocks > 1 ? (u32x4_t*)(ws + l.sums) : nullptr;
  x.pairs = (u32x4_t*)(ws + l.pairs);
  x.missed_rows = (unsigned long long*)(ws + l.missed_rows);
  x.missed_sums = (unsigned long long*)(ws + l.missed_sums);
  x.logits = (float*)(ws + l.logits);
  x.token = call_token();
  x.split_keys = pl.split_keys;
  decode_wait(x.spin_limit, x.poll_sleep);
  x.spin_limit = min(x.spin_limit, pl.polls);
  done = true;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (l.cleared && (hipStreamIsCapturing(st, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone)) {
    (void)hipGetLastError();
    const int64_t n = (int64_t)(l.cleared / 16);
    hipLaunchKernelGGL(clear_kernel, dim3((unsigned)min((n + 255) / 256, (int64_t)num_cus())), dim3(256), 0, st, (u32x4_t*)ws, n);
    KVX_HIP(hipGetLastError());
  }
  return launch_columns<true>(p, x, a.D, a.kv_dtype, st);
}

}  // namespace kvx
