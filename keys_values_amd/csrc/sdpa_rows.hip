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
#include <float.h>

#include "key_blocks.h"
#include "prefill_params.h"

namespace kvx {
namespace {

constexpr int WAVES = 4;
constexpr float kNegBig = -FLT_MAX;  // running maximum before the first visible key: finite (no inf - inf), and below the logits of any key

// Two workgroups per compute unit where the accumulators (NC D / 4 registers) leave room for two blocks in flight, else one: with 32
// rows of 128 a bound of two spills the blocks of plain and 8-bit keys, 4-bit ones fit.
constexpr int per_cu(int D, int NC, bool u4) { return NC * D <= 128 || (NC * D == 256 && D == 128 && u4) ? 2 : 1; }

template <int D, int NC, int KV>
__global__ __launch_bounds__(64 * WAVES, per_cu(D, NC, kv_is_u4(KV))) void sdpa_rows_kernel(const PrefillParams p) {
  using Blocks = KeyBlocks<D, KV, false>;
  constexpr bool F16 = kv_elem_f16(KV);
  constexpr int KJ = Blocks::KJ, DPL = Blocks::DPL, CH = Blocks::CH, COLS = 16 * NC;
  constexpr int DS = D + 4;  // floats of a row in LDS: rows start 4 banks apart
  __shared__ __align__(16) float red[WAVES][COLS][DS];
  __shared__ float rml[WAVES][COLS][2];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, kg = lane >> 4;
  const int group = blockIdx.x;  // fastest: a KV head's rows and keys stay on one XCD
  const int mblk = blockIdx.y, split = blockIdx.z;
  const int b = group / p.Hkv, kvh = group % p.Hkv;

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
  auto consume = [&](Keys& x, int chunk0) {
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
    consume(ka, chunk);
    __builtin_amdgcn_sched_barrier(0);  // the loads below reuse the registers consumed above
    issue(ka, min(chunk + 2 * STRIDE, k_end - 1));
    __builtin_amdgcn_sched_barrier(0);
    consume(kb, chunk + STRIDE);
    __builtin_amdgcn_sched_barrier(0);
    chunk += 2 * STRIDE;
  }
  if (nsteps & 1) consume(ka, chunk);

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

template <int D, int NC>
int launch_dn(const PrefillParams& p, int kv, hipStream_t st) {
  const dim3 grid(p.B * p.Hkv, p.m_blocks, p.num_splits), block(64 * WAVES);
#define KVX_ROWS_CASE(KV) \
  case KV: hipLaunchKernelGGL((sdpa_rows_kernel<D, NC, KV>), grid, block, 0, st, p); break;
  switch (kv) {
    KVX_ROWS_CASE(KVX_KV_U8)
    KVX_ROWS_CASE(KVX_KV_U4)
    KVX_ROWS_CASE(KVX_KV_U8_F16)
    KVX_ROWS_CASE(KVX_KV_U4_F16)
    default:
      if constexpr (D <= 128) {
        if (kv == KVX_KV_F16) hipLaunchKernelGGL((sdpa_rows_kernel<D, NC, KVX_KV_F16>), grid, block, 0, st, p);
        else hipLaunchKernelGGL((sdpa_rows_kernel<D, NC, KVX_KV_BF16>), grid, block, 0, st, p);
      }
  }
#undef KVX_ROWS_CASE
  KVX_HIP(hipGetLastError());
  return KVX_OK;
}

}  // namespace

namespace {

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
  int64_t step_ns = a.D == 64 ? 900 : a.D == 128 ? 1300 : 2600;
  if (plain) step_ns = step_ns * 77 / 100;
  if (columns == 32) step_ns = step_ns * (a.D == 64 ? 135 : 150) / 100;
  const int64_t ends_ns = (columns == 16 ? 1000 : 2000) * a.D / 128;
  RowsPlan best = {0, 0, INT64_MAX};
  int64_t best_per = 0;
  for (int64_t n = 1; n <= min(steps, (int64_t)64); ++n) {
    const int64_t per = (steps + n - 1) / n;
    if ((steps + per - 1) / per != n) continue;
    const int64_t c = (wgs * n + cus - 1) / cus;
    const int64_t walk = (per * step_ns + ends_ns) * (per_unit == 2 ? 180 * (c / 2) + 100 * (c % 2) : 100 * c) / 100;
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

int launch_sdpa_rows(const PrefillParams& p, int D, int kv, hipStream_t st) {
  if (D == 64) return p.columns == 16 ? launch_dn<64, 1>(p, kv, st) : launch_dn<64, 2>(p, kv, st);
  if (D == 128) return p.columns == 16 ? launch_dn<128, 1>(p, kv, st) : launch_dn<128, 2>(p, kv, st);
  return p.columns == 16 ? launch_dn<256, 1>(p, kv, st) : launch_dn<256, 2>(p, kv, st);
}

}  // namespace kvx
