// Per-key score-sums W[b,h,k] = (1/G) sum_{i,g} exp2(c * q_{i,g}.k - lse2[b,i,h*G+g]) over the visible
// (query, key) pairs, for gfx950.
//
// Reference behaviour: keys_values/attention/flashinfer_wrapper.py:51-150 (_score_sum_kernel) and
// :156-273 (host side, division by the group size); the value it must equal is
// keys_values/attention/base.py:707-725 (mean over the group, sum over queries).
//
// Key-stationary: a wavefront keeps the K rows of its 64 keys in registers as MFMA B operands for
// the whole kernel and owns those 64 outputs, so W needs no atomics and is bit-reproducible. The
// G*q_len packed query rows (row r = query r / G, head r % G) stream through LDS in tiles of 64 rows,
// double-buffered, shared by the four or eight wavefronts of the workgroup (256 or 512 keys per workgroup).
// S = Q K^T is computed with rows along M, so a lane owns one key column: the sum over queries is a
// per-lane running sum and the two halves of the wavefront are added once at the end.
// Two further kernels take short chunks: score_sum_short_kernel (few rows, few keys) and score_sum_stream_kernel (few
// rows, many keys); both can also combine the partial outputs that the attention kernel's KV splits left.
#include <type_traits>

#include "prefill_merge.h"

namespace kvx {
namespace {

constexpr int BQ = 64;    // query rows per LDS tile
constexpr int NW = 64;    // keys per wavefront
// Wavefronts per workgroup, a template argument W: 8 (512 keys per workgroup, one workgroup per compute unit: the
// Q tile staged into LDS serves twice the keys, 4 % on the kernel) or 4 (256 keys, two workgroups per compute unit); see
// score_plan.

struct ScoreParams {
  const uint16_t* q;
  const void* k;
  const float* k_scale;
  const int32_t* k_zp;
  const int32_t* tp;
  const float* lse;
  float* w;
  float* part;           // query rows split over several workgroups: (splits, B, Hkv, kv_len) partial sums, else NULL
  int32_t tiles_per_z;   // query tiles per split
  int32_t rows_per_tile; // see tile_rows
  int32_t B, Hq, Hkv, G, q_len, kv_len, R, input_pos;
  float c, inv_g;
  int64_t q_sb, q_sh, q_st, k_sb, k_sh, k_st, qs_sb, qs_sh, tp_sb, tp_sh;
};

// Q tile in LDS: [row][16-byte chunk], rows unpadded (what the global -> LDS transfer writes: a wavefront
// instruction fills 1024 contiguous bytes), chunk c of row r stored at position c ^ swz(r). The operand reads
// (ds_read_b128, 16 consecutive rows and the same chunk per phase) then touch every bank once.
template <int CPR>
__device__ __forceinline__ int swz(int r) { return CPR >= 16 ? (r & 15) : ((r >> 1) & 7); }

// Where the log-sum-exps come from the pairs of the attention's KV splits (MERGE): the most tiles a workgroup may walk, their log-sum-exps all in LDS.
// (Tables of 8192 rows leave no room for workgroups of other streams' kernels on a unit: two layers of a stack with its score-sums on
// a second stream 5.26 -> 5.48 ms. A table filled again every 32 tiles keeps its arguments alive in the loop: 40.9 -> 45 us of scattered slots' masked tiles.)
constexpr int LT = 32;

template <int D, bool MERGE>
struct alignas(16) Smem {
  static constexpr int CPR = D / 8;  // 16-byte chunks per row
  u32x4_t q[2][BQ][CPR];
  float lse[MERGE ? LT : 2][BQ];  // MERGE: of all tiles (fill_lse), +inf where a tile has no row; else a tile's are in registers before the barrier that frees its Q buffer
  int32_t qpos[4][BQ];  // read through the whole step (only by tiles that need the mask): a ring of four
};

// Rows of a tile: as many whole queries as its BQ rows hold (G = 7: 63, G = 12: 60), the rest of the tile stays empty. Every
// row then keeps its head from tile to tile and the steady steps serve any group size; with full tiles a group that does not
// divide 64 went through the general step, bounds checks and mask on every tile (attention with weights, 2 x 4 KV heads, 4096 rows
// of 7 heads over 5001 keys 168 -> 157 us; 2 x 8, 4096 rows of 3 heads over 6000 333 -> 322). Where that would leave
// more than an eighth of the tile empty (G = 24), and beyond 64 heads, tiles are full and the general step does it.
constexpr int tile_rows(int G) { return G <= BQ && BQ / G * G >= BQ - BQ / 8 ? BQ / G * G : BQ; }

// Streams the packed query rows (row r = query r / G, head r % G) of one (batch, KV head) pair into LDS, tile by
// tile, with global -> LDS transfers: no registers hold the rows on their way. Wavefront w issues instructions
// w, w + W, ... of the CPR that make a tile (RPW = 64 / CPR rows each); lane l of instruction i fills LDS position
// l % CPR of row i RPW + l / CPR, so it fetches the chunk that belongs there under the swizzle. Addresses are a
// uniform base plus a 32-bit byte offset per lane (the host checks the range). Wavefront 0 also fetches the rows'
// log-sum-exps (4 bytes per lane; MERGE: fill_lse) and writes their positions.
//   issue_steady: the tile is one of whole queries and full. Every row keeps its head and moves by BQ / G
//     queries from tile to tile: the base advances by scalar adds and the lane offsets stay.
//   issue: any tile. The offsets are formed per lane from the row's (query, head); rows past the end re-read the
//     last valid row.
//   land() overwrites the log-sum-exps of the rows a tile leaves empty and of those past the end with +inf: their weight
//     is exactly zero.
template <int D, int W, bool MERGE>
struct QLoader {
  static constexpr int CPR = D / 8;
  static constexpr int RPW = 64 / CPR;
  static constexpr int NI = CPR / W;      // transfers per wavefront and tile
  static constexpr int TILE_BYTES = BQ * CPR * 16;
  const char* qbase;   // (b, first head of the group)
  const char* lbase;   // lse + b * q_len * Hq + kvh * G
  const char* qtile;   // issue_steady: qbase advanced to the tile it fetches next
  const char* ltile;   // likewise for the log-sum-exps
  uint32_t voff0[NI];  // issue_steady: byte offset of this lane's chunk of instruction i relative to qtile
  uint32_t loff0;      // likewise for the log-sum-exp of row `lane`
  int qpv;             // likewise the position of row `lane`
  uint32_t cb[NI];     // byte offset of the chunk inside a row
  int rin[NI];         // row inside the tile
  uint32_t q_shb, q_stb, qstep, lstep;
  float inv_g;         // 1 / G: (int)((r + 0.5f) * inv_g) == r / G for the small r of a tile
  int G, R, RT, Hq, input_pos, dq, dg, wave, lane;
  int q0, g0;          // (query, head) of the first row of the next tile to fetch
  uint32_t lds_qw, lds_lse;
  int next_row0;       // first row of the next tile to fetch

  // steady_first: index (counted from row_start) of the first tile issue_steady will be asked for
  __device__ __forceinline__ void init(const ScoreParams& p, Smem<D, MERGE>& sm, int b, int kvh, int tid, int row_start, int steady_first) {
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    lane = tid & 63;
    G = p.G; R = p.R; RT = p.rows_per_tile; Hq = p.Hq; input_pos = p.input_pos;
    q_shb = (uint32_t)p.q_sh * 2u; q_stb = (uint32_t)p.q_st * 2u;
    qbase = (const char*)(p.q + b * p.q_sb + (int64_t)(kvh * p.G) * p.q_sh);
    lbase = (const char*)(p.lse + (int64_t)b * p.q_len * p.Hq + kvh * p.G);
    dq = RT / G; dg = RT % G;
    inv_g = 1.0f / (float)G;
    qstep = (uint32_t)dq * q_stb;
    lstep = (uint32_t)(dq * Hq) * 4u;
    q0 = row_start / G;
    g0 = row_start % G;
    const int qs = q0 + steady_first * dq;        // dg == 0: row_start is a multiple of RT, hence of G
    qtile = qbase + (uint64_t)qs * q_stb;
    ltile = lbase + (uint64_t)(qs * Hq) * 4u;
    qpv = input_pos + qs + lane / G;
    lds_qw = __builtin_amdgcn_readfirstlane(lds_addr_of(&sm.q[0][0][0]) + (uint32_t)(wave * 1024));
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      rin[i] = (wave + W * i) * RPW + lane / CPR;
      cb[i] = (uint32_t)(((lane % CPR) ^ swz<CPR>(rin[i])) * 16);
      const int rt = min(rin[i], RT - 1);  // the rows a tile leaves empty re-read its last one
      voff0[i] = (uint32_t)(rt % G) * q_shb + (uint32_t)(rt / G) * q_stb + cb[i];
    }
    lds_lse = __builtin_amdgcn_readfirstlane(lds_addr_of(&sm.lse[0][0]));
    const int lt = min(lane, RT - 1);
    loff0 = (uint32_t)((lt / G) * Hq + lt % G) * 4u;
    next_row0 = row_start;
  }

  template <int BUF, int I = 0>
  __device__ __forceinline__ void dma_q_steady() {
    dma16_at<(uint32_t)(BUF * TILE_BYTES + W * I * 1024)>(qtile, voff0[I], lds_qw);
    if constexpr (I + 1 < NI) dma_q_steady<BUF, I + 1>();
  }
  template <int BUF>
  __device__ __forceinline__ void issue_steady(Smem<D, MERGE>& sm, int ring) {
    dma_q_steady<BUF>();
    if (wave == 0) {
      if constexpr (!MERGE) dma4_at<(uint32_t)(BUF * BQ * 4)>(ltile, loff0, lds_lse);
      sm.qpos[ring][lane] = qpv;
      qpv += dq;
    }
    qtile += qstep;
    ltile += lstep;
    q0 += dq;
    next_row0 += RT;
  }

  // start the transfers of the next tile into Q buffer `buf` and position buffer `ring`
  __device__ __forceinline__ void issue(Smem<D, MERGE>& sm, int buf, int ring) {
    const int row0 = next_row0;
    const int rl = R - 1;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int r = min(g0 + rin[i] + q0 * G, rl) - q0 * G;  // row relative to (q0, head 0), clamped to the last valid row
      const int dqi = (int)(((float)r + 0.5f) * inv_g);         // r / G, r < G + BQ
      dma16(qbase, (uint32_t)(r - dqi * G) * q_shb + (uint32_t)(q0 + dqi) * q_stb + cb[i], lds_qw + (uint32_t)(buf * TILE_BYTES + W * i * 1024));
    }
    if (wave == 0) {
      const bool ok = row0 + lane < R;
      const int r = min(g0 + lane + q0 * G, rl) - q0 * G;
      const int dqi = (int)(((float)r + 0.5f) * inv_g);
      if constexpr (!MERGE) dma4(lbase, (uint32_t)((q0 + dqi) * Hq + (r - dqi * G)) * 4u, lds_lse + (uint32_t)(buf * BQ * 4));
      sm.qpos[ring][lane] = ok ? input_pos + q0 + dqi : INT_MAX;
    }
    q0 += dq;
    g0 += dg;
    if (g0 >= G) {
      g0 -= G;
      q0 += 1;
    }
    next_row0 = row0 + RT;
  }

  // after s_waitcnt vmcnt(0), before the barrier that publishes the tile whose first row is row0
  __device__ __forceinline__ void land(Smem<D, MERGE>& sm, int row0, int buf) const {
    if (!MERGE && wave == 0 && (lane >= RT || row0 + lane >= R)) sm.lse[buf][lane] = INFINITY;  // exp2(... - inf) = 0
  }
};

// The base-2 log-sum-exp of a row from the S (maximum, sum) pairs of its KV splits at ml[s * total_rows], shared out over T neighbouring lanes
// (a power of two; `part`: which of them this one is). Up to 16 T pairs are one memory latency.
__device__ __forceinline__ float combined_lse(const f32x2_t* ml, int64_t total_rows, int S, int part, int T) {
  float M = -INFINITY, L = 0.0f;
  for (int s0 = part; s0 < S; s0 += 16 * T) {
    f32x2_t x[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) x[u] = ml[(int64_t)min(s0 + u * T, S - 1) * total_rows];
    float Mn = M;
#pragma unroll
    for (int u = 0; u < 16; ++u) Mn = fmaxf(Mn, x[u][0]);
    const float Mu = Mn == -INFINITY ? 0.0f : Mn;
    L *= fast_exp2(M - Mu);
    M = Mn;
#pragma unroll
    for (int u = 0; u < 16; ++u) L += s0 + u * T < S ? x[u][1] * fast_exp2(x[u][0] - Mu) : 0.0f;
  }
  float Mr = M;
  for (int off = 1; off < T; off <<= 1) Mr = fmaxf(Mr, __shfl_xor(Mr, off, 64));
  const float Mu = Mr == -INFINITY ? 0.0f : Mr;
  L *= fast_exp2(M - Mu);
  for (int off = 1; off < T; off <<= 1) L += __shfl_xor(L, off, 64);
  return Mu + fast_log2(L);
}

// The log-sum-exps of the rows of `tiles` tiles from row0 on, by a workgroup of THREADS, from the pairs of the attention's KV splits. A combination
// ahead of this launch is 5 to 9 us and its gap; every workgroup working its rows' pairs out again is a latency beside that of its
// keys: 16 pairs a thread are in flight. Up to 16 pairs are added in the order of the combination (merge_rows_job), and the weights have the bits that
// its log-sum-exps give; of 17 to 32, the most (score_sum_merges), two lanes add every other one each, and the last bit may differ.
template <int THREADS>
__device__ __forceinline__ void fill_lse(const ScoreParams& p, const MergeParams& m, int b, int kvh, int tid, int row0, int tiles, float* lse_sh) {
  const int S = m.num_splits * m.teams, RT = p.rows_per_tile, n = tiles * BQ;
  const int64_t total_rows = (int64_t)p.B * p.Hkv * p.R;
  const f32x2_t* ml = (const f32x2_t*)m.part_ml + (int64_t)(b * p.Hkv + kvh) * p.R;
  auto row_of = [&](int i) { return row0 + i / BQ * RT + i % BQ; };
  auto has_row = [&](int i) { return i % BQ < RT && row_of(i) < p.R; };
  auto rows = [&](auto pairs_tag) {  // up to PAIRS pairs a row, N rows at a time
    constexpr int PAIRS = decltype(pairs_tag)::value, N = 16 / PAIRS;
    for (int i0 = tid; i0 < n; i0 += N * THREADS) {
      f32x2_t x[N][PAIRS];
#pragma unroll
      for (int u = 0; u < N; ++u)
#pragma unroll
        for (int k = 0; k < PAIRS; ++k) x[u][k] = ml[(int64_t)min(k, S - 1) * total_rows + min(row_of(i0 + u * THREADS), p.R - 1)];
#pragma unroll
      for (int u = 0; u < N; ++u) {
        const int i = i0 + u * THREADS;
        float M = x[u][0][0], L = 0.0f;
#pragma unroll
        for (int k = 1; k < PAIRS; ++k) M = fmaxf(M, x[u][k][0]);
        const float Mu = M == -INFINITY ? 0.0f : M;
#pragma unroll
        for (int k = 0; k < PAIRS; ++k) L += k < S ? x[u][k][1] * fast_exp2(x[u][k][0] - Mu) : 0.0f;
        if (i < n) lse_sh[i] = has_row(i) ? Mu + fast_log2(L) : INFINITY;
      }
    }
  };
  if (S <= 4) {
    rows(std::integral_constant<int, 4>{});
  } else if (S <= 8) {
    rows(std::integral_constant<int, 8>{});
  } else {
    const int lt = S <= 16 ? 0 : 1, T = 1 << lt, part = tid & (T - 1);
    for (int i = tid >> lt; i < n; i += THREADS >> lt) {  // the lanes of a row leave the loop together
      const float lse = combined_lse(ml + min(row_of(i), p.R - 1), total_rows, S, part, T);
      if (part == 0) lse_sh[i] = has_row(i) ? lse : INFINITY;
    }
  }
}

// QSPLIT: the query rows are split over blockIdx.z (short caches that would otherwise leave compute units
// idle); every split writes its sums to p.part and a second kernel adds them in a fixed order.
// MERGE: the attention's KV splits are still to be combined. That second kernel does it, or, without splits of the query rows, workgroups behind those of
// the key_blocks blocks of keys (merge_beside).
//
// The kernel is bound by the number of instructions a wavefront issues per tile (two wavefronts per SIMD issue
// about one instruction per ten cycles each, whatever its kind), so the tile loop comes in three forms: tiles that
// need the position mask and tiles that do not, each unrolled by two with every LDS address an immediate and the
// transfers of the tile after next sent without bounds checks ("steady"), and a general form for the last tiles.
template <int D, int KV, int W, bool QSPLIT, bool MERGE>
__global__ __launch_bounds__(64 * W, D <= 128 ? 2 : 1) void score_sum_kernel(const ScoreParams p, const MergeParams m, const int key_blocks) {
  constexpr int BK = NW * W;  // keys per workgroup
  constexpr bool F16 = kv_elem_f16(KV);  // element type of q and k
  if constexpr (MERGE && !QSPLIT) {
    if ((int)blockIdx.y >= key_blocks) {
      const int64_t job = ((int64_t)((int)blockIdx.y - key_blocks) * gridDim.x + blockIdx.x) * (W / 4);
      merge_job<D, F16, 1>(m, job + threadIdx.x / 256, threadIdx.x % 256);
      return;
    }
  }
  __shared__ Smem<D, MERGE> sm;
  __shared__ uint32_t arrivals[W];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int n = lane & 31;
  const int h = lane >> 5;
  const int group = blockIdx.x;  // fastest: (b, kvh), keeps one KV head's Q stream on one XCD
  const int b = group / p.Hkv, kvh = group % p.Hkv;
  const int key0 = blockIdx.y * BK + wave * NW;

  // K fragments (B operand): lane holds key column n of tile nt, d = 16 j + 8 h .. +8
  u32x4_t kf[2][D / 16];
  int32_t tpk[2];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const int key = key0 + nt * 32 + n;
    const bool ok = key < p.kv_len;
    tpk[nt] = ok ? (p.tp ? p.tp[b * p.tp_sb + kvh * p.tp_sh + key] : key) : INT_MAX;
    if constexpr (kv_is_plain(KV)) {
      const uint16_t* kp = (const uint16_t*)p.k + b * p.k_sb + kvh * p.k_sh + (int64_t)key * p.k_st;
#pragma unroll
      for (int j = 0; j < D / 16; ++j) {
        u32x4_t t = ok ? *(const u32x4_t*)(kp + 16 * j + 8 * h) : u32x4_t{0, 0, 0, 0};
        kf[nt][j] = t;
      }
    } else {
      const uint8_t* kp = (const uint8_t*)p.k + b * p.k_sb + kvh * p.k_sh + (int64_t)key * p.k_st;
      const int64_t so = b * p.qs_sb + kvh * p.qs_sh + key;
      const float sc = ok ? p.k_scale[so] : 0.0f;
      const int32_t zp = ok ? p.k_zp[so] : 0;
#pragma unroll
      for (int j = 0; j < D / 16; ++j) {
        u32x2_t cc;
        if constexpr (kv_is_u4(KV)) {  // chunk 2j + h of the row: one nibble of 8 bytes
          cc = ok ? *(const u32x2_t*)(kp + u4_byte_off<D>(2 * j + h)) : u32x2_t{0, 0};
          cc = u4_codes(cc, u4_shift<D>(2 * j + h));
        } else {
          cc = ok ? *(const u32x2_t*)(kp + 16 * j + 8 * h) : u32x2_t{0, 0};
        }
        kf[nt][j] = dequant_words<F16>(cc[0], cc[1], zp, sc);
      }
    }
  }
  // Largest position among this wavefront's keys: query tiles whose smallest position is at least
  // that need no mask at all (true for every key written before the current chunk).
  int tpmax = max(tpk[0], tpk[1]);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) tpmax = max(tpmax, __shfl_xor(tpmax, off, 64));
  tpmax = __builtin_amdgcn_readfirstlane(tpmax);

  float wacc[2] = {0.0f, 0.0f};
  const int tbase = QSPLIT ? (int)blockIdx.z * p.tiles_per_z : 0;  // first query tile of this workgroup
  const int RT = p.rows_per_tile;
  const int num_qt = QSPLIT ? min(p.tiles_per_z, (p.R + RT - 1) / RT - tbase) : (p.R + RT - 1) / RT;
  // Steps [0, t_steady) are steady: tiles are of whole queries and tiles t + 1 and t + 2 exist and are full.
  // Steps [0, t_masked) need the mask: the first query position of tile t, input_pos + (tbase + t) RT / G, is below
  // the largest key position of this wavefront. Both are even, so the buffer index stays a compile-time constant.
  const int nfull = min(num_qt, p.R / RT - tbase);
  const int t_steady = (RT % p.G == 0) ? (max(nfull - 2, 0) & ~1) : 0;
  int t_masked;
  {
    const int64_t need = (int64_t)max(min(tpmax, p.input_pos + p.q_len) - p.input_pos, 0) * p.G;  // rows whose position is below tpmax
    const int64_t tiles = (need + RT - 1) / RT - tbase;
    t_masked = (int)max((int64_t)0, min(tiles, (int64_t)num_qt));
    t_masked = min((t_masked + 1) & ~1, t_steady);
  }
  QLoader<D, W, MERGE> ld;
  ld.init(p, sm, b, kvh, tid, tbase * RT, 2);
  // LDS byte offsets of this lane's Q fragments (A operand): row mt 32 + n, chunk 2 j + h at position chunk ^ swz(row)
  constexpr int CPR = D / 8;
  uint32_t qa[D / 16];
#pragma unroll
  for (int j = 0; j < D / 16; ++j) qa[j] = (uint32_t)((n * CPR + ((2 * j + h) ^ swz<CPR>(n))) * 16);

  // The Q fragments of a block (32 query rows, A operand) and the rows' log-sum-exps are requested together, ahead
  // of the block's first matrix instruction: the reads then have the previous block's tail to arrive in. BUF is a
  // compile-time constant, so every read is one address register plus an immediate offset.
  auto load_q = [&](u32x4_t (&qq)[D / 16], auto buf_tag, auto mt_tag) {
    constexpr int BUF = decltype(buf_tag)::value, MT = decltype(mt_tag)::value;
    const char* qb = (const char*)&sm.q[BUF][MT * 32][0];
#pragma unroll
    for (int j = 0; j < D / 16; ++j) qq[j] = *(const u32x4_t*)(qb + qa[j]);
  };
  // accumulator rows of a lane are 8 a + 4 h + (0..3)
  auto load_lse = [&](f32x4_t (&ls)[4], int t, auto buf_tag, auto mt_tag) {
    constexpr int BUF = decltype(buf_tag)::value, MT = decltype(mt_tag)::value;
    const float* l = &sm.lse[MERGE ? t : BUF][4 * h];
#pragma unroll
    for (int a = 0; a < 4; ++a) ls[a] = *(const f32x4_t*)(l + MT * 32 + 8 * a);
  };
  // S block = 32 query rows x 64 keys, K in registers; k-steps J0 .. J1 - 1
  auto mfma_part = [&](f32x16_t (&s)[2], const u32x4_t (&qq)[D / 16], auto j0_tag, auto j1_tag) {
#pragma unroll
    for (int j = decltype(j0_tag)::value; j < decltype(j1_tag)::value; ++j) {
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        if (j == 0) {
          const f32x16_t zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
          s[nt] = mfma_32x32x16<F16>(qq[j], kf[nt][j], zero);
        } else {
          s[nt] = mfma_32x32x16<F16>(qq[j], kf[nt][j], s[nt]);
        }
      }
    }
  };
  // p = exp2(c S - lse) summed over the block's rows, quarters A0 .. A1 - 1
  auto valu_part = [&](auto mask_tag, const f32x16_t (&s)[2], const f32x4_t (&ls)[4], int ring, int mt, auto a0_tag, auto a1_tag) {
    constexpr bool MASK = decltype(mask_tag)::value;
#pragma unroll
    for (int a = decltype(a0_tag)::value; a < decltype(a1_tag)::value; ++a) {
      int4 qp = {0, 0, 0, 0};
      if constexpr (MASK) qp = *(const int4*)&sm.qpos[ring][mt * 32 + 8 * a + 4 * h];
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        float e0 = fast_exp2(fmaf(s[nt][4 * a + 0], p.c, -ls[a][0]));
        float e1 = fast_exp2(fmaf(s[nt][4 * a + 1], p.c, -ls[a][1]));
        float e2 = fast_exp2(fmaf(s[nt][4 * a + 2], p.c, -ls[a][2]));
        float e3 = fast_exp2(fmaf(s[nt][4 * a + 3], p.c, -ls[a][3]));
        if constexpr (MASK) {
          e0 = tpk[nt] > qp.x ? 0.0f : e0;
          e1 = tpk[nt] > qp.y ? 0.0f : e1;
          e2 = tpk[nt] > qp.z ? 0.0f : e2;
          e3 = tpk[nt] > qp.w ? 0.0f : e3;
        }
        wacc[nt] += (e0 + e1) + (e2 + e3);
      }
    }
  };
  // one matrix instruction, then its share of the other block's vector work (6 or 10 instructions per matrix
  // instruction, 2 of them transcendental)
  auto interleave = [&](auto mask_tag, auto quarters_tag) {
    constexpr bool MASK = decltype(mask_tag)::value;
#pragma unroll
    for (int a = 0; a < decltype(quarters_tag)::value; ++a) {
      if constexpr (MASK) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // the positions of rows 8 a .. 8 a + 7
#pragma unroll
      for (int i = 0; i < (D / 16) / 2; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, MASK ? 8 * 16 / (2 * (D / 16)) : 4 * 16 / (2 * (D / 16)), 0);
        __builtin_amdgcn_sched_group_barrier(0x400, 2 * 16 / (2 * (D / 16)), 0);
      }
    }
  };

  // Keeps a half step's work in that half: without a use here the optimiser moves the exponentials of several
  // half steps below the matrix instructions of the next ones (out of their shadow, and every block's scores then
  // need registers of their own).
  auto pin = [&](f32x16_t (&s)[2]) {
    asm volatile("" : "+v"(s[0]), "+v"(s[1]), "+v"(wacc[0]), "+v"(wacc[1]));
  };
  constexpr std::integral_constant<int, 0> I0{};
  constexpr std::integral_constant<int, 1> I1{};
  constexpr std::integral_constant<int, 3> I3{};
  constexpr std::integral_constant<int, 4> I4{};
  constexpr std::integral_constant<int, D / 16> KS{};
  constexpr std::integral_constant<int, D / 16 * 3 / 4> KS3{};
  // The workgroup's barrier, once a tile, in two halves: a wavefront arrives, in a word of LDS, when its transfers have landed and what it needs of the
  // tile is in registers, and looks for the others behind the last quarter of that block's work. As one barrier (us): 4096 rows over 8 x 32768 keys
  // 289 -> 283 of 760, 600 over 16 x 6000 30.8 -> 29.2, of 64 over 8 x 16384 123 -> 116. All wavefronts of a workgroup are resident and arrive once a tile, so the wait ends.
  uint32_t due = 0;
  auto arrive = [&] {
    ++due;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __hip_atomic_store(&arrivals[wave], due, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  auto wait_for_all = [&] {
    while (__any(__hip_atomic_load(&arrivals[lane % W], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < due)) {
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  };
  if (tid < W) arrivals[tid] = 0;
  ld.issue(sm, 0, 0);
  if (num_qt > 1) ld.issue(sm, 1, 1);
  f32x16_t sa[2], sb[2];  // blocks 0 and 1 of the current tile
  u32x4_t qq[D / 16];

  // Software pipeline: the matrix work of one block runs under the vector work of the block before.
  // Tile t + 2 is requested right behind the barrier of step t (the buffers of tile t are free from there on: its
  // Q rows have been multiplied and its log-sum-exps are in registers), has the rest of that step and the first
  // half of the next to arrive, and is published by the barrier of step t + 1.
  auto step = [&](auto mask_tag, auto steady_tag, auto buf_tag, int t) {
    constexpr bool STEADY = decltype(steady_tag)::value;
    constexpr int BUF = decltype(buf_tag)::value;
    constexpr std::integral_constant<int, BUF ^ 1> NEXT{};
    const int ring = t & 3;
    const bool more = STEADY || t + 1 < num_qt;
    f32x4_t ls[4], ls1[4];
    load_q(qq, buf_tag, I1);
    load_lse(ls, t, buf_tag, I0);
    __builtin_amdgcn_sched_barrier(0);
    mfma_part(sb, qq, I0, KS3);
    valu_part(mask_tag, sa, ls, ring, 0, I0, I3);
    interleave(mask_tag, I3);
    pin(sb);
    __builtin_amdgcn_sched_barrier(0);
    load_lse(ls1, t, buf_tag, I1);  // into registers before the barrier that hands the buffer to tile t + 2
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wavefront's part of tile t + 1 has landed
    if (!MERGE && (!STEADY || RT < BQ)) {
      if (more) ld.land(sm, (tbase + t + 1) * RT, BUF ^ 1);
    }
    arrive();
    __builtin_amdgcn_sched_barrier(0);
    mfma_part(sb, qq, KS3, KS);
    valu_part(mask_tag, sa, ls, ring, 0, I3, I4);
    interleave(mask_tag, I1);
    pin(sb);
    __builtin_amdgcn_sched_barrier(0);
    wait_for_all();
    if constexpr (STEADY) {
      ld.template issue_steady<BUF>(sm, (t + 2) & 3);
    } else {
      if (t + 2 < num_qt) ld.issue(sm, BUF, (t + 2) & 3);
    }
    if (more) {
      load_q(qq, NEXT, I0);
      __builtin_amdgcn_sched_barrier(0);
      mfma_part(sa, qq, I0, KS);
      valu_part(mask_tag, sb, ls1, ring, 1, I0, I4);
      interleave(mask_tag, I4);
      pin(sa);
      __builtin_amdgcn_sched_barrier(0);
    } else {
      valu_part(mask_tag, sb, ls1, ring, 1, I0, I4);
    }
  };
  constexpr std::true_type YES{};
  constexpr std::false_type NO{};
  if constexpr (MERGE) fill_lse<64 * W>(p, m, b, kvh, tid, tbase * RT, num_qt, &sm.lse[0][0]);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the K fragments and the first tiles have arrived
  ld.land(sm, tbase * RT, 0);
  if (num_qt > 1) ld.land(sm, (tbase + 1) * RT, 1);
  __syncthreads();
  load_q(qq, I0, I0);
  mfma_part(sa, qq, I0, KS);
  int t = 0;
  for (; t < t_masked; t += 2) {
    step(YES, YES, I0, t);
    step(YES, YES, I1, t + 1);
  }
  for (; t < t_steady; t += 2) {
    step(NO, YES, I0, t);
    step(NO, YES, I1, t + 1);
  }
  // the last tiles (and all of them when G does not divide the tile height): masked whether they need it or not
  for (; t + 1 < num_qt; t += 2) {
    step(YES, NO, I0, t);
    step(YES, NO, I1, t + 1);
  }
  if (t < num_qt) step(YES, NO, I0, t);

#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const float tot = sum_halves(wacc[nt]);
    const int key = key0 + nt * 32 + n;
    if (h == 0 && key < p.kv_len) {
      if constexpr (QSPLIT) p.part[(((int64_t)blockIdx.z * p.B + b) * p.Hkv + kvh) * p.kv_len + key] = tot;
      else p.w[((int64_t)b * p.Hkv + kvh) * p.kv_len + key] = tot * p.inv_g;
    }
  }
}

// The base-2 log-sum-exps and positions of the rows of nblk blocks of 32, in LDS, by a workgroup of 256; rows past the end
// weigh nothing. With KV splits (m.num_splits > 1) from their (maximum, sum) pairs, else from p.lse. A pass over 16 splits is a memory
// latency of 1 to 2 us; few rows share a row's splits out over up to eight neighbouring lanes.
__device__ __forceinline__ void row_weights(const ScoreParams& p, const MergeParams& m, int b, int kvh, int nblk, float* lse_sh, int32_t* qpos_sh) {
  const float inv_G = 1.0f / (float)p.G;
  const int S = m.num_splits * m.teams, group = b * p.Hkv + kvh;
  const int64_t total_rows = (int64_t)p.B * p.Hkv * p.R;
  const int lt = nblk <= 1 ? 3 : nblk <= 2 ? 2 : nblk <= 4 ? 1 : 0, T = 1 << lt, part = threadIdx.x & (T - 1);
  for (int r = threadIdx.x >> lt; r < nblk * 32; r += 256 >> lt) {  // the lanes of a row leave the loop together
    const int rc = min(r, p.R - 1), qi = (int)(((float)rc + 0.5f) * inv_G);
    float lse;
    if (m.num_splits <= 1) {
      lse = p.lse[((int64_t)b * p.q_len + qi) * p.Hq + kvh * p.G + (rc - qi * p.G)];
    } else {
      lse = combined_lse((const f32x2_t*)m.part_ml + (int64_t)group * p.R + rc, total_rows, S, part, T);
    }
    if (part == 0) {
      lse_sh[r] = r < p.R ? lse : INFINITY;
      qpos_sh[r] = p.input_pos + qi;
    }
  }
}

// Short chunks: the same sums with the query rows split over the four wavefronts of a workgroup instead of streamed past
// each of them. A workgroup owns 64 keys, held by every wavefront as B operands; wavefront w takes the 32-row blocks w,
// w + 4, ... straight from memory (the next block's rows are fetched while one is worked on, no LDS, no barriers in the
// loop), and the four sums are added in order at the end. What bounds the kernel above on few rows is its serial walk: a
// wavefront meets every tile of 64 rows, about 1 us each, whatever the number of keys, with a barrier a tile; here the walk is a
// quarter as long and a workgroup four (eight) times as small, and the partials of the attention kernel's KV splits are
// combined in the same launch: the first workgroups take 64 keys each and work out the rows' log-sum-exps from the splits'
// (maximum, sum) pairs for themselves, the others write the outputs. Rows are read from the L2 once per 64 keys instead of
// once per 256 or 512, which is why many rows keep the kernel above.
constexpr int SHORT_ROWS = 1024;  // rows whose log-sum-exps and positions the workgroup keeps in LDS

template <int D, int KV, int SC>
__global__ __launch_bounds__(256, D <= 128 ? 2 : 1) void score_sum_short_kernel(const ScoreParams p, const MergeParams m, const int score_jobs) {
  constexpr bool F16 = kv_elem_f16(KV);
  constexpr int KS = D / 16;
  if ((int)blockIdx.x >= score_jobs) {
    merge_job<D, F16, SC>(m, (int)blockIdx.x - score_jobs, threadIdx.x);
    return;
  }
  __shared__ __align__(16) float lse_sh[SHORT_ROWS];
  __shared__ __align__(16) int32_t qpos_sh[SHORT_ROWS];
  __shared__ float red[4][NW];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31;
  const int h = lane >> 5;
  const int groups = p.B * p.Hkv;
  const int group = blockIdx.x % groups;  // fastest: a KV head's query rows stay on one XCD
  const int b = group / p.Hkv, kvh = group % p.Hkv;
  const int key0 = (int)blockIdx.x / groups * NW;
  const float inv_G = 1.0f / (float)p.G;  // (int)((r + 0.5f) * inv_G) == r / G for the r < 1024 of a chunk
  auto query_of = [&](int r) { return (int)(((float)r + 0.5f) * inv_G); };
  const uint16_t* qbase = p.q + b * p.q_sb + (int64_t)(kvh * p.G) * p.q_sh;

  // Q fragments (A operand) of a block of 32 rows: lane holds row n, d = 16 j + 8 h .. +8; rows past the end re-read the last one
  auto load_q = [&](u32x4_t (&qq)[KS], int blk) {
    const int r = min(blk * 32 + n, p.R - 1);
    const int qi = query_of(r);
    const uint16_t* qp = qbase + (int64_t)(r - qi * p.G) * p.q_sh + (int64_t)qi * p.q_st + 8 * h;
#pragma unroll
    for (int j = 0; j < KS; ++j) qq[j] = *(const u32x4_t*)(qp + 16 * j);
  };
  const int nblk = (p.R + 31) / 32;
  u32x4_t qa[KS], qb[KS];
  load_q(qa, min(wave, nblk - 1));

  // K fragments (B operand): lane holds key column n of tile nt, d = 16 j + 8 h .. +8; keys past the end re-read the last
  // one (nothing of theirs is stored)
  u32x4_t kf[2][KS];
  int32_t tpk[2];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const int key = min(key0 + nt * 32 + n, p.kv_len - 1);
    tpk[nt] = p.tp ? p.tp[b * p.tp_sb + kvh * p.tp_sh + key] : key;
    if constexpr (kv_is_plain(KV)) {
      const uint16_t* kp = (const uint16_t*)p.k + b * p.k_sb + kvh * p.k_sh + (int64_t)key * p.k_st + 8 * h;
#pragma unroll
      for (int j = 0; j < KS; ++j) kf[nt][j] = *(const u32x4_t*)(kp + 16 * j);
    } else {
      const uint8_t* kp = (const uint8_t*)p.k + b * p.k_sb + kvh * p.k_sh + (int64_t)key * p.k_st;
      const int64_t so = b * p.qs_sb + kvh * p.qs_sh + key;
      const float sc = p.k_scale[so];
      const int32_t zp = p.k_zp[so];
#pragma unroll
      for (int j = 0; j < KS; ++j) {
        u32x2_t cc;
        if constexpr (kv_is_u4(KV)) cc = u4_codes(*(const u32x2_t*)(kp + u4_byte_off<D>(2 * j + h)), u4_shift<D>(2 * j + h));
        else cc = *(const u32x2_t*)(kp + 16 * j + 8 * h);
        kf[nt][j] = dequant_words<F16>(cc[0], cc[1], zp, sc);
      }
    }
  }

  row_weights(p, m, b, kvh, nblk, lse_sh, qpos_sh);
  int tpmax = max(tpk[0], tpk[1]);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) tpmax = max(tpmax, __shfl_xor(tpmax, off, 64));
  tpmax = __builtin_amdgcn_readfirstlane(tpmax);
  __syncthreads();

  float wacc[2] = {0.0f, 0.0f};
  auto block = [&](const u32x4_t (&qq)[KS], int blk) {
    f32x16_t s[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[nt][i] = 0.0f;
#pragma unroll
    for (int j = 0; j < KS; ++j)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) s[nt] = mfma_32x32x16<F16>(qq[j], kf[nt][j], s[nt]);
    const bool masked = tpmax > p.input_pos + query_of(blk * 32);
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const f32x4_t ls = *(const f32x4_t*)&lse_sh[blk * 32 + 8 * a + 4 * h];
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        float e[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = fast_exp2(fmaf(s[nt][4 * a + i], p.c, -ls[i]));
        if (masked) {
          const int4 qp = *(const int4*)&qpos_sh[blk * 32 + 8 * a + 4 * h];
          e[0] = tpk[nt] > qp.x ? 0.0f : e[0];
          e[1] = tpk[nt] > qp.y ? 0.0f : e[1];
          e[2] = tpk[nt] > qp.z ? 0.0f : e[2];
          e[3] = tpk[nt] > qp.w ? 0.0f : e[3];
        }
        wacc[nt] += (e[0] + e[1]) + (e[2] + e[3]);
      }
    }
  };
  for (int blk = wave; blk < nblk; blk += 8) {
    if (blk + 4 < nblk) load_q(qb, blk + 4);
    block(qa, blk);
    if (blk + 4 < nblk) {
      if (blk + 8 < nblk) load_q(qa, blk + 8);
      block(qb, blk + 4);
    }
  }
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const float t = sum_halves(wacc[nt]);
    if (h == 0) red[wave][nt * 32 + n] = t;
  }
  __syncthreads();
  if (tid < NW && key0 + tid < p.kv_len)
    p.w[(int64_t)group * p.kv_len + key0 + tid] = (((red[0][tid] + red[1][tid]) + red[2][tid]) + red[3][tid]) * p.inv_g;
}

// Few rows over many keys: the rows stay in LDS and the keys stream past. The tiled kernel meets a new
// workgroup of keys with a memory latency for its keys, another for its first tile and two barriers a tile, for two tiles of
// work (8 x 65536 keys of 128, 32 to 128 rows: 54 us, 2.5 TB/s). Here a wavefront walks blocks of 64 keys, the next block's
// rows in flight to registers while one is multiplied by all query rows, without barriers; as in the short kernel the partials
// of the attention's KV splits are combined by the first workgroups of the same launch. Bound by the read of K.
constexpr int stream_rows(int D) { return D <= 128 ? 256 : 128; }

template <int D, int KV, int SC>
__global__ __launch_bounds__(256, D <= 128 ? 2 : 1) void score_sum_stream_kernel(const ScoreParams p, const MergeParams m, const int merge_jobs, const int wgs_per_group) {
  constexpr bool F16 = kv_elem_f16(KV), PLAIN = kv_is_plain(KV), U4 = kv_is_u4(KV);
  constexpr int KS = D / 16, CPR = D / 8, ROWS = stream_rows(D);
  if ((int)blockIdx.x < merge_jobs) {
    merge_job<D, F16, SC>(m, (int)blockIdx.x, threadIdx.x);
    return;
  }
  __shared__ u32x4_t q_sh[ROWS][CPR];  // chunk c of row r at c ^ swz(r)
  __shared__ __align__(16) float lse_sh[ROWS];
  __shared__ __align__(16) int32_t qpos_sh[ROWS];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31;
  const int h = lane >> 5;
  const int job = (int)blockIdx.x - merge_jobs, groups = p.B * p.Hkv;
  const int group = job % groups;  // fastest: a KV head's query rows stay on one XCD
  const int b = group / p.Hkv, kvh = group % p.Hkv;
  const float inv_G = 1.0f / (float)p.G;
  const int nblk = (p.R + 31) / 32, nkb = (p.kv_len + NW - 1) / NW;

  // a block of 64 keys (B operand): lane holds key column n of tile nt, d = 16 j + 8 h .. +8; keys past the end re-read
  // the last one (nothing of theirs is stored)
  struct Keys {
    u32x4_t k[PLAIN ? 2 : 1][PLAIN ? KS : 1];
    u32x2_t c[PLAIN ? 1 : 2][PLAIN ? 1 : (U4 ? KS / 2 : KS)];
    int32_t tp[2], zp[2];
    float sc[2];
  };
  const char* kbase = (const char*)p.k + (b * p.k_sb + kvh * p.k_sh) * (PLAIN ? 2 : 1);
  const int64_t so = b * p.qs_sb + kvh * p.qs_sh;
  const int32_t* tpb = p.tp ? p.tp + b * p.tp_sb + kvh * p.tp_sh : nullptr;
  auto load_k = [&](Keys& x, int kb) {
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int key = min(kb * NW + nt * 32 + n, p.kv_len - 1);
      const char* kp = kbase + (int64_t)key * p.k_st * (PLAIN ? 2 : 1);
      x.tp[nt] = tpb ? tpb[key] : key;
      if constexpr (PLAIN) {
#pragma unroll
        for (int j = 0; j < KS; ++j) x.k[nt][j] = *(const u32x4_t*)(kp + 32 * j + 16 * h);
      } else {
        x.sc[nt] = p.k_scale[so + key];
        x.zp[nt] = p.k_zp[so + key];
#pragma unroll
        for (int j = 0; j < (U4 ? KS / 2 : KS); ++j) x.c[nt][j] = *(const u32x2_t*)(kp + (U4 ? u4_byte_off<D>(2 * j + h) : (uint32_t)(16 * j + 8 * h)));
      }
    }
  };
  const int stride = 4 * wgs_per_group;
  int kb = job / groups * 4 + wave;
  Keys ka, kc;
  if (kb < nkb) load_k(ka, kb);

  for (int i = tid; i < nblk * 32 * CPR; i += 256) {
    const int r = i / CPR, c = i % CPR, rc = min(r, p.R - 1), qi = (int)(((float)rc + 0.5f) * inv_G);
    q_sh[r][c ^ swz<CPR>(r)] = *(const u32x4_t*)(p.q + b * p.q_sb + (int64_t)(kvh * p.G + rc - qi * p.G) * p.q_sh + (int64_t)qi * p.q_st + 8 * c);
  }
  row_weights(p, m, b, kvh, nblk, lse_sh, qpos_sh);
  __syncthreads();

  auto weigh = [&](const u32x4_t (&kf)[2][KS], const int32_t (&tpk)[2], int kb) {
    float wacc[2] = {0.0f, 0.0f};
    const int tpm = max(tpk[0], tpk[1]);
    for (int blk = 0; blk < nblk; ++blk) {
      f32x16_t s[2];
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[nt][i] = 0.0f;
#pragma unroll
      for (int j = 0; j < KS; ++j) {
        const u32x4_t qq = q_sh[blk * 32 + n][(2 * j + h) ^ swz<CPR>(n)];
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) s[nt] = mfma_32x32x16<F16>(qq, kf[nt][j], s[nt]);
      }
      const bool masked = __any(tpm > p.input_pos + (int)(((float)(blk * 32) + 0.5f) * inv_G));
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const f32x4_t ls = *(const f32x4_t*)&lse_sh[blk * 32 + 8 * a + 4 * h];
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          float e[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) e[i] = fast_exp2(fmaf(s[nt][4 * a + i], p.c, -ls[i]));
          if (masked) {
            const int4 qp = *(const int4*)&qpos_sh[blk * 32 + 8 * a + 4 * h];
            e[0] = tpk[nt] > qp.x ? 0.0f : e[0];
            e[1] = tpk[nt] > qp.y ? 0.0f : e[1];
            e[2] = tpk[nt] > qp.z ? 0.0f : e[2];
            e[3] = tpk[nt] > qp.w ? 0.0f : e[3];
          }
          wacc[nt] += (e[0] + e[1]) + (e[2] + e[3]);
        }
      }
    }
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const float t = sum_halves(wacc[nt]);
      const int key = kb * NW + nt * 32 + n;
      if (h == 0 && key < p.kv_len) p.w[(int64_t)group * p.kv_len + key] = t * p.inv_g;
    }
  };
  if constexpr (PLAIN) {
    for (; kb < nkb; kb += 2 * stride) {
      const bool more = kb + stride < nkb;
      if (more) load_k(kc, kb + stride);
      weigh(ka.k, ka.tp, kb);
      if (more) {
        if (kb + 2 * stride < nkb) load_k(ka, kb + 2 * stride);
        weigh(kc.k, kc.tp, kb + stride);
      }
    }
  } else {
    for (; kb < nkb; kb += stride) {
      u32x4_t kf[2][KS];
      const int32_t tpk[2] = {ka.tp[0], ka.tp[1]};
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int j = 0; j < KS; ++j) {
          u32x2_t cc = ka.c[nt][U4 ? j % (KS / 2) : j];
          if constexpr (U4) cc = u4_codes(cc, u4_shift<D>(2 * j + h));
          kf[nt][j] = dequant_words<F16>(cc[0], cc[1], ka.zp[nt], ka.sc[nt]);
        }
      if (kb + stride < nkb) load_k(ka, kb + stride);
      weigh(kf, tpk, kb);
    }
  }
}

// What a split of the query rows leaves behind, in one launch: the first merge_jobs workgroups combine the attention's KV splits, the others add the
// splits' sums, W = (1/G) * (part[0] + part[1] + ...), in that order.
template <int D, bool F16>
__global__ __launch_bounds__(256) void score_sum_finish_kernel(const MergeParams m, const int merge_jobs, const float* part, float* w, int pairs, int kv_len, int splits, float inv_g) {
  if ((int)blockIdx.x < merge_jobs) {
    merge_job<D, F16, 1>(m, blockIdx.x, threadIdx.x);
    return;
  }
  // pairs fastest: on the die whose L2 has the pair's sums
  const uint32_t job = blockIdx.x - merge_jobs, at = job / (uint32_t)pairs, key = at * 256 + threadIdx.x;
  if (key >= (uint32_t)kv_len) return;
  const int64_t n = (int64_t)pairs * kv_len, i = (int64_t)(job - at * pairs) * kv_len + key;
  float acc = part[i];
  for (int z = 1; z < splits; ++z) acc += part[(int64_t)z * n + i];
  w[i] = acc * inv_g;
}

// Wavefronts per workgroup and splits of the query rows with the least estimated time. c workgroups share a compute unit: of
// four wavefronts two run side by side, of eight (and at head size 256 of four) one; a full count with a nearly empty last round
// is what the estimate avoids. Measured constants (ns, head size 128): a tile of 64 rows takes a pair of workgroups 2600, one alone
// 1500, a workgroup of eight wavefronts 2500; its keys cost a workgroup 3000 before the first tile; the launch that adds
// the splits' sums 4000 and its reads at 4 TB/s. Against splits to two workgroups a unit, each of 8 tiles or more (attention with
// weights, us): 8 KV heads x 4096 keys, 600 rows 44.3 -> 40.8, x 10000 keys, 4096 rows 261 -> 255; 4 x 6000 keys of 256, 600 / 1500
// rows 73 -> 62, 123 -> 108.
struct ScorePlan {
  int splits, tiles_per_z, waves;
};
ScorePlan score_plan(const kvx_sdpa_args& a) {
  const int G = a.Hq / a.Hkv, RT = tile_rows(G);
  const int num_qt = (int)(((int64_t)a.q_len * G + RT - 1) / RT);
  const int64_t groups = (int64_t)a.B * a.Hkv, cus = num_cus(), scale = a.D;  // of the tiles' and keys' times: D / 128
  const int64_t wgs = groups * ((a.kv_len + 4 * NW - 1) / (4 * NW)), wide = groups * ((a.kv_len + 8 * NW - 1) / (8 * NW));
  ScorePlan best = {1, num_qt, 4};
  int64_t best_ns = INT64_MAX;
  auto consider = [&](int splits, int waves) {
    const int64_t tiles = (num_qt + splits - 1) / splits;
    splits = (int)((num_qt + tiles - 1) / tiles);
    const bool pairs = waves == 4 && a.D <= 128;
    const int64_t c = ((waves == 8 ? wide : wgs * splits) + cus - 1) / cus;
    const int64_t walk = pairs ? tiles * (2600 * (c / 2) + 1500 * (c % 2)) + 3000 * ((c + 1) / 2) : c * (tiles * (waves == 8 ? 2500 : 1500) + 3000);
    const int64_t ns = walk * scale / 128 + (splits > 1 ? 4000 + splits * groups * a.kv_len / 1000 : 0);
    if (ns < best_ns) {
      best_ns = ns;
      best = {splits, (int)tiles, waves};
    }
  };
  if (a.D <= 128) consider(1, 8);
  for (int s = 1; s <= min(16, (num_qt + 1) / 2); ++s) consider(s, 4);
  return best;
}

// Few rows over few keys take the short kernel: 64 keys a workgroup then still leave one compute unit a workgroup, and the
// wavefronts that walk the query rows side by side would idle otherwise. Attention with weights, us, long -> short kernel:
// 2 KV heads x 1024 keys of 64, 128 / 512 / 1024 / 2000 rows 16.0 -> 12.3, 23.7 -> 17.3, 26.5 -> 24.2, 30.9 -> 37.9; 8 x 1024 of 128,
// the same rows 23.4 -> 21.2, 34.9 -> 27.7, 39.9 -> 36.4, 46.2 -> 53.8. With more keys every wavefront of the long kernel
// has work of its own and reads a quarter of the query rows: 8 x 4096 of 128, 512 rows 38.1 -> 42.5.
bool is_short(const kvx_sdpa_args& a) {
  return (int64_t)a.q_len * (a.Hq / a.Hkv) <= SHORT_ROWS && (int64_t)a.B * a.Hkv * ((a.kv_len + NW - 1) / NW) <= num_cus();
}

// The combination runs at the score jobs' occupancy, two workgroups a compute unit in the streaming kernel: more jobs than
// compute units are quicker in a launch of their own (8 x 4096 keys of 128, 32 / 128 rows: 20.6 -> 16.3 and 27 -> 34 us combined).
bool merge_fits(const kvx_sdpa_args& a) {
  const int per_job = merge_rows(a.D, merge_classes(a.D));
  return ((int64_t)a.B * a.Hq * a.q_len + per_job - 1) / per_job <= num_cus();
}
// Where the streaming kernel is the faster one: one block of rows, up to four of rows of 64 values whose splits it can combine,
// and any number it holds over 256 K keys or more; over fewer a wavefront has no second block of keys to fetch ahead.
// Attention with weights, us, tiled -> streamed: 8 x 4096 keys of 128, 32 / 64 / 128 rows 20.6 -> 16.3, 23.2 -> 24.2, 27 -> 30;
// 8 x 65536, 32 / 128 / 256 rows 99 -> 87, 126 -> 112, 150 -> 143; of 64, 4 x 9001, 128 rows 27 -> 22, 8 x 16384, 64 / 128 rows
// 27 -> 24, 28 -> 29; 16 x 20000 of 256, 32 / 128 rows 190 -> 163, 216 -> 196.
bool is_streamed(const kvx_sdpa_args& a) {
  const int64_t rows = (int64_t)a.q_len * (a.Hq / a.Hkv);
  if (is_short(a) || rows > stream_rows(a.D)) return false;
  return rows <= 32 || (a.D == 64 && rows <= 128 && merge_fits(a)) || (int64_t)a.B * a.Hkv * a.kv_len >= 256 * 1024;
}

template <int D, int KV>
int launch_t(const ScoreParams& p, int splits, int waves, const MergeParams* rest, int kind, hipStream_t st) {
  const int groups = p.B * p.Hkv;
  if (kind == KVX_SCORE_SUM_SHORT) {
    const int64_t score_jobs = (int64_t)groups * ((p.kv_len + NW - 1) / NW);
    const MergeParams m = rest ? *rest : MergeParams{};
    auto launch = [&](auto sc_tag) {
      constexpr int SC = decltype(sc_tag)::value;
      const int64_t merge_jobs = m.num_splits > 1 ? merge_blocks(m, D, SC) : 0;
      hipLaunchKernelGGL((score_sum_short_kernel<D, KV, SC>), dim3((unsigned)(score_jobs + merge_jobs)), dim3(256), 0, st, p, m, (int)score_jobs);
    };
    if (merge_wants_classes(m, D)) launch(std::integral_constant<int, merge_classes(D)>{});
    else launch(std::integral_constant<int, 1>{});
    KVX_HIP(hipGetLastError());
    return KVX_OK;
  }
  if (kind == KVX_SCORE_SUM_STREAMED) {
    const MergeParams m = rest ? *rest : MergeParams{};
    const int nkb = (p.kv_len + NW - 1) / NW, most = (nkb + 3) / 4;
    const int per_group = max(1, min(most, (D <= 128 ? 2 : 1) * num_cus() / groups));
    auto launch = [&](auto sc_tag) {
      constexpr int SC = decltype(sc_tag)::value;
      const int64_t merge_jobs = m.num_splits > 1 ? merge_blocks(m, D, SC) : 0;
      hipLaunchKernelGGL((score_sum_stream_kernel<D, KV, SC>), dim3((unsigned)(merge_jobs + (int64_t)groups * per_group)), dim3(256), 0, st, p, m, (int)merge_jobs,
                         per_group);
    };
    if (merge_wants_classes(m, D)) launch(std::integral_constant<int, merge_classes(D)>{});
    else launch(std::integral_constant<int, 1>{});
    KVX_HIP(hipGetLastError());
    return KVX_OK;
  }
  const MergeParams m = rest ? *rest : MergeParams{};
  const int64_t jobs = m.num_splits > 1 ? merge_blocks(m, D, 1) : 0;
  auto tiled = [&](auto waves_tag, auto split_tag, auto merge_tag) {
    constexpr int W = decltype(waves_tag)::value;
    constexpr bool QSPLIT = decltype(split_tag)::value, MERGE = decltype(merge_tag)::value;
    const int key_blocks = (p.kv_len + W * NW - 1) / (W * NW), per_y = groups * (W / 4);
    const dim3 grid(groups, key_blocks + (unsigned)(QSPLIT ? 0 : (jobs + per_y - 1) / per_y), splits);
    hipLaunchKernelGGL((score_sum_kernel<D, KV, W, QSPLIT, MERGE>), grid, dim3(64 * W), 0, st, p, m, key_blocks);
  };
  auto tiled_any = [&](auto waves_tag, auto split_tag) {
    if (jobs) tiled(waves_tag, split_tag, std::true_type{});
    else tiled(waves_tag, split_tag, std::false_type{});
  };
  if (splits > 1) {
    tiled_any(std::integral_constant<int, 4>{}, std::true_type{});
    KVX_HIP(hipGetLastError());
    const int64_t sums = (int64_t)groups * ((p.kv_len + 255) / 256);
    hipLaunchKernelGGL((score_sum_finish_kernel<D, kv_elem_f16(KV)>), dim3((unsigned)(jobs + sums)), dim3(256), 0, st, m, (int)jobs, p.part, p.w, groups, p.kv_len, splits,
                       p.inv_g);
  } else {
    bool wide = false;
    if constexpr (D <= 128) wide = waves == 8;
    if constexpr (D <= 128) {
      if (wide) tiled_any(std::integral_constant<int, 8>{}, std::false_type{});
    }
    if (!wide) tiled_any(std::integral_constant<int, 4>{}, std::false_type{});
  }
  KVX_HIP(hipGetLastError());
  return KVX_OK;
}

// Where the score-sums' partial sums go: the workspace, but not over partials of the attention that are still to be combined. NULL: no room.
float* score_scratch(const kvx_sdpa_args& a, const MergeParams* rest) {
  const size_t need = score_sum_workspace(a);
  if (!a.workspace || ((uintptr_t)a.workspace & 15)) return nullptr;
  size_t at = 0;
  if (rest && rest->num_splits > 1) {
    const char* ml_end = (const char*)(rest->part_ml + (size_t)2 * rest->num_splits * rest->teams * rest->B * rest->Hkv * rest->R);
    if ((size_t)((const char*)rest->part_o - (const char*)a.workspace) < need) at = ((size_t)(ml_end - (const char*)a.workspace) + 15) & ~(size_t)15;
  }
  return a.workspace_bytes >= at + need ? (float*)((char*)a.workspace + at) : nullptr;
}

// Whether workgroups beside the score jobs combine the attention's partials: the jobs' last round leaves `spare` places, for the time of a walk, and a
// workgroup takes 2.5 us there. Where they do not fit they end behind the score jobs, a few to a unit, and a launch of their own ahead is shorter. Attention with
// weights, us, launch ahead -> beside: 600 rows over 16 x 6000 keys 74 -> 71, 404 over 8 x 9444 50.3 -> 46.2, 564 of 64 over 8 x 6138 36.6 -> 33.6, 140 over
// 16 x 2443 29.9 -> 24.0. Combined in the launch that adds the sums of a split of the query rows: 460 over 8 x 4238 50.1 -> 43.7, 1716 of 64 over
// 8 x 1800 41.9 -> 35.3, 434 of 64 over 32 x 1216 35.7 -> 28.3, 2331 scattered over 8 x 5001 107.0 -> 105.6.
bool merge_beside(const kvx_sdpa_args& a, const ScorePlan& pl, const MergeParams& m) {
  const int64_t groups = (int64_t)a.B * a.Hkv, places = (int64_t)num_cus() * (pl.waves == 4 && a.D <= 128 ? 2 : 1);
  const int64_t wgs = groups * ((a.kv_len + pl.waves * NW - 1) / (pl.waves * NW)), spare = (places - wgs % places) % places;
  const int64_t jobs = merge_blocks(m, a.D, 1) / (pl.waves / 4);
  const int64_t walk = ((int64_t)pl.tiles_per_z * (pl.waves == 8 ? 2500 : 1500) + 3000) * a.D / 128;
  return jobs * 2500 <= spare * walk;
}

// Whether the score jobs' workgroups have few enough pairs to read between them, of all splits of their rows each (fill_lse): at 56 KB per us and unit (fitted over 420
// calls, 0.7 us beside it) they spend on it what a launch of its own takes, 3 us, from about 24 K pairs a unit on. Attention with weights, us, combined here -> in a
// launch of its own: up to 2500 pairs a unit 6 % longer in the mean, 10 to 12 K 2, 15 to 20 K alike; 1092 rows of 64 over 4 x 52480 keys (46 K) 147.0 -> 141.3,
// 896 of 128 over 4 x 46790 (88 K) 157.1 -> 145.5, 1336 of 64 over 4 x 45027 (118 K) 170.0 -> 152.6, 270 of 256 over 8 x 46297 (58 K) 336.8 -> 321.5. Over the 420 the
// choice takes 0.12 % longer than the better of both in the mean; always here 0.7 %, never 3.5 %.
bool pairs_are_few(const kvx_sdpa_args& a, const ScorePlan& pl, const MergeParams& m) {
  const int S = m.num_splits * m.teams, asked = S <= 4 ? 4 : S <= 8 ? 8 : S <= 16 ? 16 : 32;
  const int64_t wgs = (int64_t)a.B * a.Hkv * ((a.kv_len + pl.waves * NW - 1) / (pl.waves * NW)) * pl.splits;
  return wgs * pl.tiles_per_z * BQ * asked <= (int64_t)num_cus() * (24 << 10);
}

}  // namespace

int score_sum_kind(const kvx_sdpa_args& a) { return is_short(a) ? KVX_SCORE_SUM_SHORT : is_streamed(a) ? KVX_SCORE_SUM_STREAMED : KVX_SCORE_SUM_TILED; }
bool score_sum_combines(const kvx_sdpa_args& a) { return is_short(a) || (is_streamed(a) && merge_fits(a)); }

bool score_sum_merges(const kvx_sdpa_args& a, const MergeParams& m, bool room) {
  if (score_sum_kind(a) != KVX_SCORE_SUM_TILED || m.num_splits <= 1 || m.num_splits * m.teams > 32 || merge_wants_classes(m, a.D)) return false;
  const ScorePlan pl = score_plan(a);
  return pl.tiles_per_z <= LT && pairs_are_few(a, pl, m) && (pl.splits > 1 ? room || score_scratch(a, &m) != nullptr : merge_beside(a, pl, m));
}

size_t score_sum_workspace(const kvx_sdpa_args& a) {
  if (is_short(a) || is_streamed(a)) return 0;
  const ScorePlan pl = score_plan(a);
  return pl.splits > 1 ? (size_t)pl.splits * a.B * a.Hkv * a.kv_len * sizeof(float) : 0;
}

// The query rows are fetched at a uniform base plus a 32-bit byte offset per lane.
int check_score_sum(const kvx_sdpa_args& a) {
  const int64_t G = a.Hq / a.Hkv;
  KVX_REQUIRE(a.q_stride_h >= 0 && a.q_stride_t >= 0 && ((G - 1) * a.q_stride_h + (int64_t)(a.q_len - 1) * a.q_stride_t + a.D) * 2 < (1ll << 32),
              KVX_ERR_UNSUPPORTED, "kvx_score_sum: the query rows of one (batch, KV head) pair must span less than 4 GiB (strides %lld / %lld)",
              (long long)a.q_stride_h, (long long)a.q_stride_t);
  return KVX_OK;
}

int launch_score_sum(const kvx_sdpa_args& a, hipStream_t st, const MergeParams* rest) {
  // the query rows are split only if the caller's workspace holds the partial sums
  ScorePlan pl = score_plan(a);
  float* scratch = pl.splits > 1 ? score_scratch(a, rest) : nullptr;
  if (pl.splits > 1 && !scratch) pl = {1, 0, pl.waves};
  const int rc = check_score_sum(a);
  if (rc != KVX_OK) return rc;
  ScoreParams p;
  p.part = scratch;
  p.tiles_per_z = pl.tiles_per_z;
  p.rows_per_tile = tile_rows(a.Hq / a.Hkv);
  p.q = (const uint16_t*)a.q;
  p.k = a.k;
  p.k_scale = a.k_scale;
  p.k_zp = a.k_zp;
  p.tp = a.token_positions;
  p.lse = a.lse;
  p.w = a.w;
  p.B = a.B; p.Hq = a.Hq; p.Hkv = a.Hkv; p.G = a.Hq / a.Hkv;
  p.q_len = a.q_len; p.kv_len = a.kv_len; p.R = a.q_len * p.G; p.input_pos = a.input_pos;
  p.c = a.sm_scale * kLog2e;
  p.inv_g = 1.0f / (float)p.G;
  p.q_sb = a.q_stride_b; p.q_sh = a.q_stride_h; p.q_st = a.q_stride_t;
  p.k_sb = a.k_stride_b; p.k_sh = a.k_stride_h; p.k_st = a.k_stride_t;
  p.qs_sb = a.qs_stride_b; p.qs_sh = a.qs_stride_h;
  p.tp_sb = a.tp_stride_b; p.tp_sh = a.tp_stride_h;
  const int kind = score_sum_kind(a);
#define KVX_SCORE_SUM_CASE(KV) \
  case KV: \
    return a.D == 256 ? launch_t<256, KV>(p, pl.splits, pl.waves, rest, kind, st) : a.D == 128 ? launch_t<128, KV>(p, pl.splits, pl.waves, rest, kind, st) \
                                                                      : launch_t<64, KV>(p, pl.splits, pl.waves, rest, kind, st);
  if (a.D == 256 || a.D == 128 || a.D == 64) {
    switch (a.kv_dtype) {
      KVX_SCORE_SUM_CASE(KVX_KV_BF16)
      KVX_SCORE_SUM_CASE(KVX_KV_F16)
      KVX_SCORE_SUM_CASE(KVX_KV_U8)
      KVX_SCORE_SUM_CASE(KVX_KV_U4)
      KVX_SCORE_SUM_CASE(KVX_KV_U8_F16)
      KVX_SCORE_SUM_CASE(KVX_KV_U4_F16)
    }
  }
#undef KVX_SCORE_SUM_CASE
  return set_error(KVX_ERR_UNSUPPORTED, "kvx_score_sum: head size %d not in {64, 128, 256}", a.D);
}

}  // namespace kvx
