// Chunked-prefill attention for gfx950: O = softmax(s Q K^T + mask) V with the base-2 log-sum-exp.
//
// Reference behaviour: keys_values/attention/base.py:660-742 (eager arithmetic),
// keys_values/csrc/kernels/sdpa_prefill.cu:34-181 (what the FlashInfer prefill returns: O and
// base-2 LSE), keys_values/attention/attention_utils.py:238-247 (mask by token position).
//
// Work decomposition
//   The G query heads that share a KV head are packed into the row dimension: row r of a
//   (batch, KV head) pair is (query r / G, head r % G), R = q_len * G rows in all. A workgroup of
//   four (uint8 cache: eight) wavefronts owns 32 consecutive rows per wavefront and walks the key tiles of its KV
//   split, 64 keys at a time, so a K/V tile staged once in LDS serves all G heads.
//   Scores are produced TRANSPOSED, S^T = K Q^T (32x32x16 bf16 MFMA, keys along M, rows along N):
//   every lane then owns one row's statistics (running max and sum) and only the other half of the
//   wavefront holds the remaining keys of that row, so the online softmax needs a single
//   cross-lane exchange per tile. The accumulator layout of S^T is exactly the B-operand layout
//   of the second product O^T = V^T P^T once the 16 keys of a k-step are taken in the order
//   (0..3, 8..11 | 4..7, 12..15); the V^T operand is read from the row-major V tile with the
//   transposing LDS read (ds_read_b64_tr_b16), which delivers exactly that order.
//   K/V tiles travel global -> LDS by DMA (global_load_lds_dwordx4, no registers), double-buffered,
//   rows unpadded and XOR-swizzled against bank conflicts. The loop is software-pipelined: the
//   matrix cores add V(t-1) P(t-1) to O while the vector ALU turns S(t) into P(t).
#include <stddef.h>
#include <string.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "prefill_params.h"
#include "row_write.h"

namespace kvx {
namespace {

constexpr float kSlackLog2 = 8.0f;  // see the running-maximum update in the kernel

// Wavefronts per workgroup, 32 rows each. The uint8 cache takes 8: a tile is dequantised once per
// workgroup, so twice the rows halve that vector work per row (-13 % kernel time); for bf16 tiles the
// two sizes run alike and the smaller one leaves more workgroups for short chunks. At head size 256 the
// output accumulators (128 registers) leave no room for two wavefronts per SIMD: four for every store.
constexpr int nwaves(int kv, int D) { return (kv_is_plain(kv) || D > 128) ? 4 : 8; }  // kv: enum kvx_kv_dtype
constexpr bool pairs(int kv, int D) { return kv_is_plain(kv) && D <= 128; }  // two workgroups of a compute unit side by side

// K and V tiles in LDS: [key][16-byte chunk], rows unpadded (D * 2 bytes), chunk c of row r stored at
// position c ^ key(r). Unpadded rows are what the global -> LDS DMA writes (a wavefront fills 1024
// contiguous bytes per instruction); the XOR then has to spread what one LDS phase touches over
// the 64 banks (256 bytes per cycle; measured on gfx950 with the LDS bank-conflict counter):
//   K, ds_read_b128:        16 consecutive rows, the same chunk      -> swz_k distinct over 16 rows
//   V, ds_read_b64_tr_b16:  half a wavefront reads 4 consecutive rows x 4 chunks (64 bytes a row): rows of 256
//                           bytes or more start at the same bank, so bits 2..3 of swz_v are distinct over r % 4
//                           (with bits 1..2, as for 128-byte rows, every such read took a 2-way conflict)
// Both depend on r % 16 only, so they repeat for the row groups a wavefront loads (16 or 32 rows apart).
template <int CPR>
__device__ __forceinline__ int swz_k(int r) { return CPR >= 16 ? (r & 15) : ((r >> 1) & 7); }
template <int CPR>
__device__ __forceinline__ int swz_v(int r) { return CPR >= 16 ? (((r & 3) << 2) | ((r >> 2) & 1)) : (((r & 3) << 1) | ((r >> 2) & 1)); }

template <int D>
struct alignas(16) Smem {
  static constexpr int CPR = D / 8;  // 16-byte chunks per row
  u32x4_t k[2][BN][CPR];
  u32x4_t v[2][BN][CPR];
  int32_t tp[2][BN];  // token positions of the K tile in the buffer of the same index
};

typedef short s16x4_t __attribute__((ext_vector_type(4)));

// ds_read_b64_tr_b16: within each group of 16 lanes, lane i (a = i % 4, r = i / 4) supplies the
// address of 4 consecutive bf16 of "row r, columns 4a..4a+3"; it receives column i of rows 0..3.
typedef char __attribute__((address_space(3))) * lds_ptr_t;
__device__ __forceinline__ u32x2_t lds_read_tr16(lds_ptr_t p) {
  const s16x4_t t = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4_t __attribute__((address_space(3)))*)(p));
  return __builtin_bit_cast(u32x2_t, t);
}


// Tile loader. A wavefront instruction covers RPW = 64 / CPR whole rows; wavefront w of the
// workgroup takes row groups w, w + 4, ... of the 64-row tile (NI groups each for K and for V).
// bf16 cache: DMA into LDS. uint8 cache: codes and row state go through registers (prefetched one
// tile ahead like the DMA), are dequantised to bf16 and written to the same LDS layout.
template <int D, int KV>
struct Loader {
  static constexpr bool U8 = !kv_is_plain(KV);  // codes through registers (8-bit or 4-bit store)
  static constexpr bool U4 = kv_is_u4(KV);
  static constexpr int CPR = D / 8;
  static constexpr int RPW = 64 / CPR;        // rows per wavefront instruction: 4 (D=128), 8 (D=64)
  static constexpr int NWAVES = nwaves(KV, D);
  static constexpr int NTHREADS = 64 * NWAVES;
  static constexpr int NI = BN / RPW / NWAVES;     // instructions per wavefront per operand: 4 / 2
  static constexpr int ESZ = U8 ? 1 : 2;
  // row groups of one wavefront are NWAVES RPW rows apart: with a multiple of 16 the XOR keys, and so
  // the source chunks, are the same for all of them (not for D = 256 with four wavefronts: 8 rows)
  static constexpr bool SAME_CHUNK = (NWAVES * RPW) % 16 == 0;
  const char* kbase;
  const char* vbase;
  const float* ks;
  const int32_t* kz;
  const float* vs;
  const int32_t* vz;
  const int32_t* tp;
  int64_t k_tile_bytes, v_tile_bytes, k_st, v_st;
  int wave, lane, kv_len, rl;
  int cgk[NI], cgv[NI];         // the source chunk that belongs at this lane's LDS position, per row group
  int shk[SAME_CHUNK ? 1 : NI], shv[SAME_CHUNK ? 1 : NI];  // 4-bit store: nibble of this lane's K / V chunk (4 = high)
  uint32_t lds_k, lds_v;        // LDS addresses of the K and V buffers (wavefront-uniform)
  uint32_t lds_kw, lds_vw;      // the same plus this wavefront's row-group offset
  uint32_t koffs[NI], voffs[NI];  // byte offset of this lane's chunk of row group i inside a tile
  // uint8 path staging registers
  u32x2_t kc[NI], vc[NI];
  float ksr[NI], vsr[NI];
  int32_t kzr[NI], vzr[NI];

  __device__ __forceinline__ int row_of(int i) const { return (NWAVES * i + wave) * RPW + rl; }
  // byte offset of chunk c (8 values) inside a row
  __device__ __forceinline__ static uint32_t chunk_off(int c) { return U4 ? u4_byte_off<D>(c) : (uint32_t)(c * 8 * ESZ); }

  __device__ __forceinline__ void init(const PrefillParams& p, Smem<D>& sm, int b, int kvh, int tid) {
    lds_k = __builtin_amdgcn_readfirstlane(lds_addr_of(&sm.k[0][0][0]));
    lds_v = __builtin_amdgcn_readfirstlane(lds_addr_of(&sm.v[0][0][0]));
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wavefront-uniform: keeps the LDS targets in scalar registers
    lane = tid & 63;
    rl = lane / CPR;  // row inside the group
    kv_len = p.kv_len;
    k_st = p.k_st;
    v_st = p.v_st;
    kbase = (const char*)p.k + (b * p.k_sb + kvh * p.k_sh) * ESZ;
    vbase = (const char*)p.v + (b * p.v_sb + kvh * p.v_sh) * ESZ;
    const int64_t so = b * p.qs_sb + kvh * p.qs_sh;
    ks = p.k_scale + so;
    kz = p.k_zp + so;
    vs = p.v_scale + so;
    vz = p.v_zp + so;
    tp = p.tp ? p.tp + b * p.tp_sb + kvh * p.tp_sh : nullptr;
    k_tile_bytes = (int64_t)BN * p.k_st * ESZ;
    v_tile_bytes = (int64_t)BN * p.v_st * ESZ;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int r = row_of(i);
      cgk[i] = (lane % CPR) ^ swz_k<CPR>(r);  // the chunk that belongs at LDS position lane % CPR of row r
      cgv[i] = (lane % CPR) ^ swz_v<CPR>(r);
      if (i == 0 || !SAME_CHUNK) {
        shk[SAME_CHUNK ? 0 : i] = u4_shift<D>(cgk[i]);
        shv[SAME_CHUNK ? 0 : i] = u4_shift<D>(cgv[i]);
      }
    }
    lds_kw = lds_k + (uint32_t)(wave * RPW * CPR * 16);
    lds_vw = lds_v + (uint32_t)(wave * RPW * CPR * 16);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      koffs[i] = (uint32_t)(row_of(i) * p.k_st * ESZ + chunk_off(cgk[i]));
      voffs[i] = (uint32_t)(row_of(i) * p.v_st * ESZ + chunk_off(cgv[i]));
    }
  }

  // a full tile of the bf16 cache into buffer BUF: one scalar add (into M0) per DMA instruction
  template <bool IS_K, int BUF, int I = 0>
  __device__ __forceinline__ void issue_full(const char* tb) {
    dma16_at<(uint32_t)((BUF * BN + NWAVES * I * RPW) * CPR * 16)>(tb, IS_K ? koffs[I] : voffs[I], IS_K ? lds_kw : lds_vw);
    if constexpr (I + 1 < NI) issue_full<IS_K, BUF, I + 1>(tb);
  }
  template <bool IS_K, int BUF>
  __device__ __forceinline__ void issue_full(int tile) {
    issue_full<IS_K, BUF, 0>((IS_K ? kbase : vbase) + tile * (IS_K ? k_tile_bytes : v_tile_bytes));
  }

  template <bool IS_K>
  __device__ __forceinline__ void issue_one(Smem<D>& sm, int tile, int buf, int tid) {
    const int key0 = tile * BN;
    const int tpb = buf;
    if constexpr (!U8) {
      if (key0 + BN <= kv_len) {  // the common case: immediate LDS offsets, shared scalar base
        if (buf == 0) issue_full<IS_K, 0>(tile);
        else issue_full<IS_K, 1>(tile);
        issue_tp<IS_K>(sm, tile, tpb);
        return;
      }
    }
    const char* base = IS_K ? kbase : vbase;
    const int64_t st = IS_K ? k_st : v_st;
    const char* tb = base + tile * (IS_K ? k_tile_bytes : v_tile_bytes);
    if (key0 + BN <= kv_len) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        if constexpr (!U8) {
          const uint32_t dst = (IS_K ? lds_k : lds_v) + (uint32_t)((buf * BN + (NWAVES * i + wave) * RPW) * CPR * 16);
          dma16(tb, IS_K ? koffs[i] : voffs[i], dst);
        } else {
          const int key = key0 + row_of(i);
          const u32x2_t c = *(const u32x2_t*)(tb + (IS_K ? koffs[i] : voffs[i]));
          if (IS_K) { kc[i] = c; ksr[i] = ks[key]; kzr[i] = kz[key]; }
          else { vc[i] = c; vsr[i] = vs[key]; vzr[i] = vz[key]; }
        }
      }
    } else {
      // last, partial tile: rows past the end re-read the last valid row (finite data); their
      // position is INT_MAX, so they are masked for every query and contribute exactly zero
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int key = min(key0 + row_of(i), kv_len - 1);
        const uint32_t off = (uint32_t)((int64_t)(key - key0) * st * ESZ) + chunk_off(IS_K ? cgk[i] : cgv[i]);
        if constexpr (!U8) {
          const uint32_t dst = (IS_K ? lds_k : lds_v) + (uint32_t)((buf * BN + (NWAVES * i + wave) * RPW) * CPR * 16);
          dma16(tb, off, dst);
        } else {
          const u32x2_t c = *(const u32x2_t*)(tb + off);
          if (IS_K) { kc[i] = c; ksr[i] = ks[key]; kzr[i] = kz[key]; }
          else { vc[i] = c; vsr[i] = vs[key]; vzr[i] = vz[key]; }
        }
      }
    }
    issue_tp<IS_K>(sm, tile, tpb);
  }

  // a full tile, not the last one of the walk: no bounds to check (bf16 tiles only)
  template <bool IS_K, int BUF>
  __device__ __forceinline__ void issue_steady(Smem<D>& sm, int tile) {
    static_assert(!U8, "codes go through registers");
    issue_full<IS_K, BUF>(tile);
    if (IS_K && tp && wave == 0)
      dma4((const char*)(tp + tile * BN), (uint32_t)lane * 4, __builtin_amdgcn_readfirstlane(lds_addr_of(&sm.tp[BUF][0])));
  }
  __device__ __forceinline__ void land_steady(Smem<D>& sm, int tile, int buf, int tid) {
    if (!tp && tid < BN) sm.tp[buf][tid] = tile * BN + tid;
  }

  // token positions of the K tile: one 4-byte DMA per lane of wavefront 0 (slots past the end
  // re-read the last valid one and are overwritten with INT_MAX when the tile lands)
  template <bool IS_K>
  __device__ __forceinline__ void issue_tp(Smem<D>& sm, int tile, int buf) {
    if (IS_K && tp && wave == 0) {
      const int key0 = tile * BN;
      const uint32_t dst = lds_addr_of(&sm.tp[buf][0]);
      dma4((const char*)(tp + key0), (uint32_t)min(lane, kv_len - 1 - key0) * 4, __builtin_amdgcn_readfirstlane(dst));
    }
  }

  // make tile `tile`, issued last, visible in LDS (called after s_waitcnt vmcnt(0), before the
  // barrier that publishes it)
  template <bool IS_K>
  __device__ __forceinline__ void land(Smem<D>& sm, int tile, int buf, int tid) {
    const int tpb = buf;
    if constexpr (U8) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int r = row_of(i);
        u32x2_t c = IS_K ? kc[i] : vc[i];
        if constexpr (U4) c = u4_codes(c, IS_K ? shk[SAME_CHUNK ? 0 : i] : shv[SAME_CHUNK ? 0 : i]);
        if (IS_K) sm.k[buf][r][lane % CPR] = dequant_words<kv_elem_f16(KV)>(c[0], c[1], kzr[i], ksr[i]);
        else sm.v[buf][r][lane % CPR] = dequant_words<kv_elem_f16(KV)>(c[0], c[1], vzr[i], vsr[i]);
      }
    }
    if (IS_K && tid < BN) {
      const int key = tile * BN + tid;
      if (!tp) sm.tp[tpb][tid] = key < kv_len ? key : INT_MAX;
      else if (key >= kv_len) sm.tp[tpb][tid] = INT_MAX;
    }
  }
};

// Jobs of a causal first chunk in splits, in the order of their length. A split covers the keys of `period` blocks of rows, so that the
// rows of period i see the splits before i whole and their own in part: first all the whole ones, then the others from the longest on.
__device__ __forceinline__ void causal_job(const PrefillParams& p, int job, int& mblk, int& split) {
  const int P = p.period, n = p.num_splits, last = p.m_blocks - (n - 1) * P;  // blocks of the last period, 1 to P
  for (int i = n - 1; i > 0; --i) {
    const int blocks = i == n - 1 ? last : P;
    if (job < blocks * i) {
      mblk = i * P + job / i;
      split = job % i;
      return;
    }
    job -= blocks * i;
  }
  const int longer = (P - last) * (n - 1);  // places in a period that the last one does not have
  if (job < longer) {
    split = job % (n - 1);
    mblk = split * P + P - 1 - job / (n - 1);
  } else {
    job -= longer;
    split = job % n;
    mblk = split * P + last - 1 - job / n;
  }
}

// PERIODS: jobs of a causal first chunk in splits (causal_job; decided at run time it cost every call 0.2 us)
// PAIR: two teams of four wavefronts walk the two halves of the split for the same rows, as two workgroups of a compute unit would, and combine
// them in LDS: two splits' partials neither go through memory nor take a launch (pick_splits). The teams have barriers of their own: with the
// workgroup's barrier each waits for the other at every tile (4096 rows of 128, 8 x 32768 keys 515 us; two workgroups 483 and the merge). A
// wavefront arrives at its team's barrier, a word in LDS, with the last quarter of the second product still to issue and looks for the others
// behind it: 483 -> 477, 8 x 16384 scattered keys 272 -> 266 (two workgroups and the merge 277).
// WRITE: a first chunk whose rows the launch also writes to their slots. Each workgroup (of a row's splits the first) does so ahead of its own work for the
// tokens whose first rows it has, and clears its share of the slots behind the chunk's. The write's loads and quantisation run under
// the products of the unit's other workgroup. As a launch of its own the write of 8192 x 8 rows took 14.5 us before an attention of 503. (Behind its own
// work the same code made the compiler order the exponentials worse: 512 -> 544 us.)
struct NoWrite {};
struct FirstWrite {
  kvx_cache_write_args a;
  uint32_t rest;  // slots behind the chunk's, of a row
};

template <int D, int KV, bool PERIODS, bool PAIR, bool WRITE = false>
__global__ __launch_bounds__(64 * nwaves(KV, D) * (PAIR ? 2 : 1), (kv_is_plain(KV) && D <= 128) ? 2 : 1) void sdpa_prefill_kernel(
    const PrefillParams p, const std::conditional_t<WRITE, FirstWrite, NoWrite> wr) {
  static_assert(!WRITE || (kv_is_plain(KV) && !PAIR && nwaves(KV, D) * 64 == NTHREADS), "a first chunk's own rows");
  static_assert(!PAIR || (pairs(KV, D) && !PERIODS), "two teams fit a compute unit");
  constexpr bool F16 = kv_elem_f16(KV);  // element type of q, k, v, o
  constexpr int BM = 32 * nwaves(KV, D);  // rows per workgroup
  constexpr int CPR = D / 8;
  constexpr int KS = D / 16;  // k-steps of the first product
  constexpr int DT = D / 32;  // d tiles of the second product
  constexpr int TEAM = 64 * nwaves(KV, D);
  __shared__ Smem<D> sms[PAIR ? 2 : 1];
  const int team = PAIR ? __builtin_amdgcn_readfirstlane(threadIdx.x / TEAM) : 0;
  Smem<D>& sm = sms[team];
  __shared__ uint32_t arrivals[PAIR ? 2 : 1][4];
  const int tid = PAIR ? threadIdx.x % TEAM : threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int n = lane & 31;  // row (query) owned by this lane within the wavefront's 32 rows
  const int h = lane >> 5;  // which half of each 8-wide k group / which 4-row group of the MFMA output

  const int group = blockIdx.x;  // b * Hkv + kvh: fastest-varying so that a KV head stays on one XCD
  // slots in position order (a causal first chunk): the later rows see more tiles; they start first, so that the short
  // ones fill up the end (a first chunk of 8192 tokens, 32 heads of 128: 597 -> 543 us)
  int mblk = p.tp ? blockIdx.y : gridDim.y - 1 - blockIdx.y, split = blockIdx.z;
  if constexpr (PERIODS) causal_job(p, blockIdx.y, mblk, split);
  const int b = group / p.Hkv;
  const int kvh = group % p.Hkv;

  const int row0w = mblk * BM + wave * 32;
  const int row = row0w + n;
  const bool row_ok = row < p.R;
  const int rowc = row_ok ? row : p.R - 1;
  const int qi = rowc / p.G;
  const int g = rowc % p.G;
  const int qpos = p.input_pos + qi;
  const int qpos_min_w = p.input_pos + min(row0w, p.R - 1) / p.G;

  if constexpr (WRITE) {
    if (split == 0) {
      const kvx_cache_write_args& a = wr.a;
      const int t0 = (mblk * BM + p.G - 1) / p.G, t1 = min((mblk * BM + BM + p.G - 1) / p.G, p.q_len);
      switch (a.kv_dtype) {
        case KVX_KV_BF16:
        case KVX_KV_F16: write_tokens<D, KV>(a, b, kvh, t0, t1); break;
        case KVX_KV_U8:
        case KVX_KV_U8_F16: write_tokens<D, F16 ? KVX_KV_U8_F16 : KVX_KV_U8>(a, b, kvh, t0, t1); break;
        default: write_tokens<D, F16 ? KVX_KV_U4_F16 : KVX_KV_U4>(a, b, kvh, t0, t1);
      }
      const uint32_t total = (uint32_t)(a.B * a.Hkv) * wr.rest, step = (uint32_t)(p.B * p.Hkv * p.m_blocks) * NTHREADS;  // (below 2^31 both: checked by the host)
      for (uint32_t at = (uint32_t)(mblk * p.B * p.Hkv + group) * NTHREADS + threadIdx.x; at < total; at += step) {
        const uint32_t row = at / wr.rest;
        const int64_t to = row / a.Hkv * a.sc_stride_b + row % a.Hkv * a.sc_stride_h + a.num + (at - row * wr.rest);
        if (a.scores) a.scores[to] = 0.0f;
        if (a.v_norm) a.v_norm[to] = 0.0f;
        if (a.q_errors) a.q_errors[to] = 0.0f;
      }
    }
  }

  // Q fragments (B operand): lane holds row n, d = 16 j + 8 h .. +8
  u32x4_t qf[KS];
  {
    const uint16_t* qp = p.q + b * p.q_sb + (int64_t)(kvh * p.G + g) * p.q_sh + (int64_t)qi * p.q_st;
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      u32x4_t t = row_ok ? *(const u32x4_t*)(qp + 16 * j + 8 * h) : u32x4_t{0, 0, 0, 0};
      qf[j] = t;
    }
  }

  // LDS byte offsets of this lane's operand fragments inside a tile buffer.
  // K (A operand of S^T = K Q^T): row 32 mt + n, chunk 2 j + h, stored at position chunk ^ swz_k(row).
  uint32_t ka[KS];
#pragma unroll
  for (int j = 0; j < KS; ++j) ka[j] = (uint32_t)(n * CPR + ((2 * j + h) ^ swz_k<CPR>(n))) * 16;
  // V (A operand of O^T = V^T P^T) through the transposing read: in its group of 16 lanes this lane
  // points at key row (i / 4) + 4 h of the 16-key block and at d columns 16 * (group % 2) + 4 (i % 4) .. +3
  // of the 32-d tile; the second read of a k-step is 8 rows further down (same XOR key, same positions).
  const int li = lane & 15;
  const int vrow = (li >> 2) + 4 * h;                              // + 32 mt + 16 j (+ 8)
  const int vcol = 16 * ((lane >> 4) & 1) + 4 * (li & 3);          // + 32 dt, bf16 elements
  uint32_t va[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    const int c = (32 * dt + vcol) >> 3;
    va[dt] = (uint32_t)((vrow * CPR + (c ^ swz_v<CPR>(vrow))) * 16 + (vcol & 7) * 2);
  }

  int tile_begin = split * p.tiles_per_split;
  int tile_end = min(tile_begin + p.tiles_per_split, p.num_tiles);
  if (!p.tp) {
    // slots hold positions 0, 1, 2, ...: tiles past the last position any row of this workgroup may
    // see are masked out completely (the upper triangle of a causal first chunk) and are skipped
    const int qpos_max = p.input_pos + min(mblk * BM + BM - 1, p.R - 1) / p.G;
    tile_end = min(tile_end, qpos_max / BN + 1);
    if (tile_end <= tile_begin) {  // whole split invisible (only with num_splits > 1): its output is not read
      if (row_ok) {
        const int64_t prow = ((int64_t)(PAIR ? 2 * split + team : split) * p.B * p.Hkv + group) * p.R + row;
        if (h == 0) {
          p.part_ml[prow * 2] = -INFINITY;
          p.part_ml[prow * 2 + 1] = 0.0f;
        }
      }
      return;
    }
  }
  // The teams' halves are those of a whole split, as if each were a split of its own; the second team may be left without a tile
  if constexpr (PAIR) {
    const int half = tile_begin + (p.tiles_per_split + 1) / 2;
    if (team == 0) tile_end = min(tile_end, half);
    else tile_begin = min(half, tile_end);
  }
  const int mine = tile_end - tile_begin;

  f32x16_t o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.0f;
  float m = -INFINITY;  // reference (lazy running maximum) of the raw, unscaled scores of this row
  const float slack = kSlackLog2 / p.c;
  float l = 0.0f;       // this lane's share of the running sum

  // S^T of one tile from the K tile in k[buf]: two independent accumulator chains
  auto qk = [&](f32x16_t (&s)[2], int buf) {
    const char* kb = (const char*)&sm.k[buf][0][0];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[mt][i] = 0.0f;
#pragma unroll
    for (int j = 0; j < KS; ++j)
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        const u32x4_t kk = *(const u32x4_t*)(kb + ka[j] + mt * 32 * CPR * 16);
        s[mt] = mfma_32x32x16<F16>(kk, qf[j], s[mt]);
      }
  };
  // mask (only tiles that hold a position some row of this wavefront may not see)
  auto mask = [&](f32x16_t (&s)[2], int buf) {
    const int tpl = sm.tp[buf][lane];
    // bit k: key k of the tile holds a position some row of this wavefront may not see. In a cache with
    // scattered slots nearly every tile has a few such keys: only their groups of 8 keys are masked.
    const unsigned long long hidden = __ballot(tpl > qpos_min_w);
    if (hidden) {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          if ((hidden >> (mt * 32 + 8 * a)) & 0xffull) {
            const int4 tq = *(const int4*)&sm.tp[buf][mt * 32 + 8 * a + 4 * h];
            if (tq.x > qpos) s[mt][4 * a + 0] = -INFINITY;
            if (tq.y > qpos) s[mt][4 * a + 1] = -INFINITY;
            if (tq.z > qpos) s[mt][4 * a + 2] = -INFINITY;
            if (tq.w > qpos) s[mt][4 * a + 3] = -INFINITY;
          }
        }
    }
  };

  // second product for one tile: O^T += V^T P^T with V from v[buf]; matrix instructions FIRST ..
  // FIRST + COUNT - 1 of the 4 DT in (key block, d tile) order
  auto pv_part = [&](const uint32_t (&pb)[2][8], int buf, auto first_tag, auto count_tag) {
    constexpr int FIRST_I = decltype(first_tag)::value, COUNT = decltype(count_tag)::value;
    // one LDS pointer per d tile; every read below is that pointer plus a compile-time offset
    lds_ptr_t vl[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) vl[dt] = (lds_ptr_t)((const char*)&sm.v[buf][0][0] + va[dt]);
#pragma unroll
    for (int i = FIRST_I; i < FIRST_I + COUNT; ++i) {
      const int mt = i / (2 * DT), j = (i / DT) % 2, dt = i % DT;
      const u32x4_t pf = u32x4_t{pb[mt][4 * j], pb[mt][4 * j + 1], pb[mt][4 * j + 2], pb[mt][4 * j + 3]};
      const int rb = (32 * mt + 16 * j) * CPR * 16;
      const u32x2_t lo = lds_read_tr16(vl[dt] + rb);
      const u32x2_t hi = lds_read_tr16(vl[dt] + rb + 8 * CPR * 16);
      o[dt] = mfma_32x32x16<F16>(u32x4_t{lo[0], lo[1], hi[0], hi[1]}, pf, o[dt]);
    }
  };
  auto v_operand = [&](int buf, int i) {
    const int mt = i / (2 * DT), j = (i / DT) % 2, dt = i % DT;
    const lds_ptr_t v = (lds_ptr_t)((const char*)&sm.v[buf][0][0] + va[dt]) + (32 * mt + 16 * j) * CPR * 16;
    const u32x2_t lo = lds_read_tr16(v), hi = lds_read_tr16(v + 8 * CPR * 16);
    return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
  };
  auto pv_one = [&](const uint32_t (&pb)[2][8], int i, u32x4_t v) {
    const int mt = i / (2 * DT), j = (i / DT) % 2, dt = i % DT;
    o[dt] = mfma_32x32x16<F16>(v, u32x4_t{pb[mt][4 * j], pb[mt][4 * j + 1], pb[mt][4 * j + 2], pb[mt][4 * j + 3]}, o[dt]);
  };
  auto pv = [&](const uint32_t (&pb)[2][8], int buf) {
    pv_part(pb, buf, std::integral_constant<int, 0>{}, std::integral_constant<int, 4 * DT>{});
  };
  // The first NPRE matrix instructions of the second product go out right behind the first product:
  // they keep the matrix core busy while the vector ALU reduces the maximum of S(t), which has to wait
  // for the first product anyway.
  constexpr int NPRE = DT;

  // Pipeline: iteration t multiplies S(t) = K(t) Q^T, then lets the matrix cores add V(t-1) P(t-1)
  // to O while the vector ALU turns S(t) into P(t). K(t) sits in k[t & 1]; V(t-1) in v[(t-1) & 1];
  // K(t+1) and V(t) are in flight to the other buffers and are published by the barrier that ends
  // the iteration.
  Loader<D, KV> ld;
  ld.init(p, sm, b, kvh, tid);
  uint32_t pbs[2][2][8];  // packed P of the tile in buffer 0 / 1: written by one step, multiplied by the next
  // The team's barrier: how often each of its wavefronts has arrived. All eight wavefronts of a workgroup are resident, and each arrives once a
  // tile whatever the other team does, so a wait ends.
  uint32_t due = 0;
  if constexpr (PAIR) {
    if (threadIdx.x < 8) arrivals[threadIdx.x >> 2][threadIdx.x & 3] = 0;
    __syncthreads();
  }
  auto arrive = [&] {
    if constexpr (PAIR) {
      ++due;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      __hip_atomic_store(&arrivals[team][wave], due, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  };
  auto sync = [&] {
    if constexpr (PAIR) {
      while (__any(__hip_atomic_load(&arrivals[team][lane & 3], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < due)) {
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    } else {
      __syncthreads();
    }
  };
  // every split owns at least one tile (the host sizes the splits that way)
  if (!PAIR || mine > 0) {
    ld.template issue_one<true>(sm, tile_begin, 0, tid);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the first K tile and the Q fragments have arrived
    ld.template land<true>(sm, tile_begin, 0, tid);
    arrive();
    sync();
  }
  // one pipeline step on the tile in buffer CUR (compile time: LDS offsets become immediates and P
  // alternates between two register sets instead of being copied)
  auto step = [&](auto first_tag, auto cur_tag, auto steady_tag, int t) {
    constexpr bool FIRST = decltype(first_tag)::value;
    constexpr int cur = decltype(cur_tag)::value;
    // STEADY: tiles t and t + 1 are full and tile t + 1 belongs to this walk
    constexpr bool STEADY = decltype(steady_tag)::value && kv_is_plain(KV);
    uint32_t (&pb_prev)[2][8] = pbs[cur ^ 1];
    uint32_t (&pb)[2][8] = pbs[cur];
    const bool has1 = STEADY || t + 1 < tile_end;
    if constexpr (STEADY) {
      ld.template issue_steady<false, cur>(sm, t);
      ld.template issue_steady<true, cur ^ 1>(sm, t + 1);
    } else {
      ld.template issue_one<false>(sm, t, cur, tid);
      if (has1) ld.template issue_one<true>(sm, t + 1, cur ^ 1, tid);
    }
    // publish the tiles that were in flight
    auto publish = [&] {
      __builtin_amdgcn_s_setprio(3);
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wavefront's DMA / loads have landed
      if constexpr (STEADY) {
        ld.land_steady(sm, t + 1, cur ^ 1, tid);
      } else {
        ld.template land<false>(sm, t, cur, tid);
        if (has1) ld.template land<true>(sm, t + 1, cur ^ 1, tid);
      }
      arrive();
    };
    f32x16_t s[2];
    // Issue priority rises through the tile (0 for the first product, 1 for the dependent chain mask ->
    // maximum -> rescaling decision, 2 for the exponentials beside the second product, 3 for the way to the
    // barrier): of the two wavefronts on a SIMD the one closer to its barrier goes first, so the four
    // wavefronts of a workgroup wait less for each other. Measured -3 to -5 % on the kernel.
    __builtin_amdgcn_s_setprio(0);
    qk(s, cur);
    if constexpr (!FIRST) {
      pv_part(pb_prev, cur ^ 1, std::integral_constant<int, 0>{}, std::integral_constant<int, NPRE>{});
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(1);
    mask(s, cur);
    // ---- running maximum; rescale only when some row of the wavefront has a new maximum ------
    float mx = fmaxf(s[0][0], s[1][0]);
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(fmaxf(mx, s[0][i]), s[1][i]);
    mx = max_halves(mx);
    float alpha = 1.0f;
    // m is a reference, not the exact maximum: it moves only when a score exceeds it by 2^kSlackLog2
    // in the exponent, which keeps every p below 2^kSlackLog2 and makes rescaling rare
    const bool resc = __any(mx > m + slack);
    if (resc) {
      const float m_new = fmaxf(m, mx);
      const float m_use = (m_new == -INFINITY) ? 0.0f : m_new;
      alpha = fast_exp2((m - m_use) * p.c);
      l *= alpha;
      m = m_new;
    }
    // ---- O += V(t-1) P(t-1) on the matrix cores, P(t) = exp2(c S(t) - c m) on the vector ALU ----
    __builtin_amdgcn_s_setprio(2);
    // PAIR: the last quarter of it comes behind the arrival at the team's barrier
    constexpr int NREST = 4 * DT - NPRE, NLAST = PAIR && !FIRST ? NREST / 4 : 0;
    if constexpr (!FIRST) pv_part(pb_prev, cur ^ 1, std::integral_constant<int, NPRE>{}, std::integral_constant<int, NREST - NLAST>{});
    const float mc = (m == -INFINITY) ? 0.0f : m * p.c;
    float rs0 = 0.0f, rs1 = 0.0f;
    auto weigh = [&](int mt, int i0, int i1) {
#pragma unroll
      for (int i = i0; i < i1; i += 2) {
        const float p0 = fast_exp2(fmaf(s[mt][i], p.c, -mc));
        const float p1 = fast_exp2(fmaf(s[mt][i + 1], p.c, -mc));
        rs0 += p0;
        rs1 += p1;
        pb[mt][i >> 1] = pack_pair<F16>(p0, p1);
      }
    };
    weigh(0, 0, 16);
    weigh(1, 0, NLAST ? 8 : 16);
    if constexpr (NLAST == 0) l += rs0 + rs1;
    if constexpr (!FIRST) {
      // interleave in the instruction stream: each matrix instruction of the second product is
      // followed by the two LDS reads of the next one and by its share of the softmax arithmetic,
      // so the vector ALU works in the shadow of the matrix core instead of after it
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);  // operands of the first two go out ahead
      constexpr int NV = (80 + NREST - 1) / NREST;  // VALU per matrix instruction: 80 per tile (fma, add, cvt)
      constexpr int NX = (32 + NREST - 1) / NREST;  // transcendental: 32 exp2 per tile
#pragma unroll
      for (int i = 0; i < NREST - NLAST; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);             // 1 MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, (NV + 1) / 2, 0);  // half of its vector work,
        __builtin_amdgcn_sched_group_barrier(0x400, (NX + 1) / 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);             // the 2 LDS reads of the next one,
        __builtin_amdgcn_sched_group_barrier(0x002, NV / 2, 0);        // the other half
        __builtin_amdgcn_sched_group_barrier(0x400, NX / 2, 0);
      }
      // keep the softmax arithmetic in this block: without a use here the optimiser sinks it
      // past the barrier below, out of the matrix core's shadow
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int i = 0; i < (NLAST && mt == 1 ? 4 : 8); ++i) asm volatile("" : "+v"(pb[mt][i]));
      asm volatile("" : "+v"(l));
      if constexpr (NLAST > 0) {
        u32x4_t vl[NLAST];
#pragma unroll
        for (int i = 0; i < NLAST; ++i) vl[i] = v_operand(cur ^ 1, 4 * DT - NLAST + i);
        publish();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NLAST; ++i) pv_one(pb_prev, 4 * DT - NLAST + i, vl[i]);
        weigh(1, 8, 16);
        l += rs0 + rs1;
#pragma unroll
        for (int i = 0; i < NLAST; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, (20 + NLAST - 1) / NLAST, 0);
          __builtin_amdgcn_sched_group_barrier(0x400, (8 + NLAST - 1) / NLAST, 0);
        }
#pragma unroll
        for (int i = 4; i < 8; ++i) asm volatile("" : "+v"(pb[1][i]));
        asm volatile("" : "+v"(l));
      }
      if (resc) {  // O (now including tile t-1) moves to the new reference maximum
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
      }
    }
    if constexpr (NLAST == 0) publish();
    sync();
  };
  constexpr std::integral_constant<int, 0> B0{};
  constexpr std::integral_constant<int, 1> B1{};
  constexpr std::true_type YES{};
  constexpr std::false_type NO{};
  // A wavefront behind the last row has its share of the tiles to bring and nothing to multiply: those that have rows get the issue slots. us: 128 rows over
  // 8 x 32768 8-bit keys (four of eight wavefronts) 49.3 -> 38.6, 4-bit 51.5 -> 39.6, of 64 values 32.5 -> 26.9, 35.5 -> 26.3; 136 / 260 / 520 plain rows 40.7 -> 36.3,
  // 56.1 -> 51.7, 86.1 -> 81.7. (Of 256 values the kernel spills as it is, and with this beside it takes 1.4 times as long.)
  const bool idle = D <= 128 && __builtin_amdgcn_readfirstlane(row0w) >= p.R;
  if (D <= 128 && idle) {
    for (int t = tile_begin, cur = 0; t < tile_end; ++t, cur ^= 1) {
      const bool has1 = t + 1 < tile_end;
      ld.template issue_one<false>(sm, t, cur, tid);
      if (has1) ld.template issue_one<true>(sm, t + 1, cur ^ 1, tid);
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
      ld.template land<false>(sm, t, cur, tid);
      if (has1) ld.template land<true>(sm, t + 1, cur ^ 1, tid);
      arrive();
      sync();
    }
  } else if (!PAIR || mine > 0) {
    step(YES, B0, NO, tile_begin);
    int t = tile_begin + 1;
    // tiles whose successor is a full tile of this walk take the step without bounds checks
    const int steady_end = min(tile_end - 1, p.kv_len / BN - 1);  // t < steady_end: tiles t, t + 1 full, t + 1 < tile_end
    for (; t + 1 < steady_end; t += 2) {
      step(NO, B1, YES, t);
      step(NO, B0, YES, t + 1);
    }
    for (; t + 1 < tile_end; t += 2) {
      step(NO, B1, NO, t);
      step(NO, B0, NO, t + 1);
    }
    if (t < tile_end) {
      step(NO, B1, NO, t);
      pv(pbs[1], 1);
    } else {
      pv(pbs[0], 0);
    }
  }

  // ---- epilogue -----------------------------------------------------------------------------
  const float lt = sum_halves(l);
  if constexpr (PAIR) {
    // Each team completes half of the columns. The tiles' place holds what the other one needs: [register quad][thread], and behind it the
    // rows' maxima and sums. Products and sums are those of the combining launch, and where more splits follow the row's sum is left to it: maxima and
    // sums of both teams, as of two splits, so that the log-sum-exp does not depend on who walks a split.
    constexpr int HALF = DT / 2;
    const float mr = m * p.c;
    __syncthreads();  // the tiles have been multiplied
    f32x4_t* mail = (f32x4_t*)&sms[team];
    f32x2_t* stat = (f32x2_t*)(mail + 4 * HALF * TEAM);
    const f32x4_t* from = (const f32x4_t*)&sms[team ^ 1];
    const f32x2_t* from_stat = (const f32x2_t*)(from + 4 * HALF * TEAM);
    auto send = [&](auto first_tag) {
      constexpr int FIRST = decltype(first_tag)::value;
#pragma unroll
      for (int i = 0; i < 4 * HALF; ++i) {
        const f32x16_t& x = o[FIRST + i / 4];
        mail[i * TEAM + tid] = f32x4_t{x[4 * (i % 4)], x[4 * (i % 4) + 1], x[4 * (i % 4) + 2], x[4 * (i % 4) + 3]};
      }
    };
    if (team == 0) send(std::integral_constant<int, HALF>{});
    else send(std::integral_constant<int, 0>{});
    if (h == 0) stat[32 * wave + n] = f32x2_t{mr, lt};
    __syncthreads();
    const f32x2_t other = from_stat[32 * wave + n];
    const float M = fmaxf(mr, other[0]), Mu = M == -INFINITY ? 0.0f : M;
    const float w_own = fast_exp2(mr - Mu), w_other = fast_exp2(other[0] - Mu);
    const float L = lt * w_own + other[1] * w_other;
    const int64_t prow = ((int64_t)split * p.B * p.Hkv + group) * p.R + row;
    const float inv = L > 0.0f ? 1.0f / L : 0.0f;
    uint16_t* op = p.o + b * p.o_sb + (int64_t)(kvh * p.G + g) * p.o_sh + (int64_t)qi * p.o_st;
    auto finish = [&](auto first_tag) {
      constexpr int FIRST = decltype(first_tag)::value;
#pragma unroll
      for (int i = 0; i < 4 * HALF; ++i) {
        const f32x4_t x = from[i * TEAM + tid];
        const int dt = FIRST + i / 4, a = i % 4;
        f32x4_t y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = o[dt][4 * a + e] * w_own + x[e] * w_other;
        if (!row_ok) continue;
        if (p.num_splits == 1) *(u32x2_t*)(op + dt * 32 + 8 * a + 4 * h) = u32x2_t{pack_pair<F16>(y[0] * inv, y[1] * inv), pack_pair<F16>(y[2] * inv, y[3] * inv)};
        else *(f32x4_t*)(p.part_o + prow * D + dt * 32 + 8 * a + 4 * h) = y;
      }
    };
    if (team == 0) finish(std::integral_constant<int, 0>{});
    else finish(std::integral_constant<int, HALF>{});
    if (h == 0 && row_ok) {
      if (p.num_splits > 1) *(f32x2_t*)(p.part_ml + (((int64_t)(2 * split + team) * p.B * p.Hkv + group) * p.R + row) * 2) = f32x2_t{mr, lt};
      else if (p.lse && team == 0) p.lse[((int64_t)b * p.q_len + qi) * p.Hq + kvh * p.G + g] = Mu + fast_log2(L);
    }
    return;
  }
  if (p.num_splits == 1) {
    const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
    if (row_ok) {
      uint16_t* op = p.o + b * p.o_sb + (int64_t)(kvh * p.G + g) * p.o_sh + (int64_t)qi * p.o_st;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          u32x2_t w2;
          w2[0] = pack_pair<F16>(o[dt][4 * a] * inv, o[dt][4 * a + 1] * inv);
          w2[1] = pack_pair<F16>(o[dt][4 * a + 2] * inv, o[dt][4 * a + 3] * inv);
          *(u32x2_t*)(op + dt * 32 + 8 * a + 4 * h) = w2;
        }
      if (p.lse && h == 0) p.lse[((int64_t)b * p.q_len + qi) * p.Hq + kvh * p.G + g] = m * p.c + fast_log2(lt);
    }
  } else {
    if (row_ok) {
      const int64_t prow = ((int64_t)split * p.B * p.Hkv + group) * p.R + row;
      float* po = p.part_o + prow * D;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          f32x4_t w4 = {o[dt][4 * a], o[dt][4 * a + 1], o[dt][4 * a + 2], o[dt][4 * a + 3]};
          *(f32x4_t*)(po + dt * 32 + 8 * a + 4 * h) = w4;
        }
      if (h == 0) {
        p.part_ml[prow * 2] = m * p.c;  // -inf if the split saw no visible key
        p.part_ml[prow * 2 + 1] = lt;
      }
    }
  }
}

template <int D, bool F16, int SC>
__global__ __launch_bounds__(256) void sdpa_prefill_merge_kernel(const MergeParams p) { merge_job<D, F16, SC>(p, blockIdx.x, threadIdx.x); }

// The number of KV splits with the least estimated time, and whether a split is walked by a pair of teams (PAIR): c workgroups share a compute
// unit, one after the other or side by side, and each walks its split's tiles; more splits balance the device better and shorten the walk, but
// every partial is written, read again and combined by one more launch. Constants in ns: a tile of 64 keys for a workgroup that has its compute unit
// to itself 840 / 1130 / 2050 at head size 64 / 128 / 256; at 128 two workgroups side by side take 1.48 of that, an odd one after them 1.06; at 64
// two 1.46 and three, all that run side by side, 1.95, one and two after them 1.13 and 1.41; a pair takes 1.45, 1.6 with others after it, of 64 1.5,
// for two tiles and needs no partials where the split is the only one. Workgroups over codes or of head size 256 run one after the other.
// Over 450 calls of 40 to 1100 rows of 1 to 8 heads, 4 to 1100 blocks of rows, 500 to 40000 keys, the plan chosen takes 0.5 % longer than the best of up to 30
// in the mean, the best plan without pairs 6 %. us, best without pairs -> with: 80 blocks x 13 tiles 24.8 -> 20.0, 120 x 13 27.9 -> 20.4,
// 32 x 94 30.7 -> 27.1, 60 x 396 of 64 values 77.3 -> 72.8; 256 x 64 90.8 -> 78, x 256 277 -> 266, x 512 483 -> 477. A full count of rounds with a nearly
// empty last one is what the rule avoids: 2 x 4 heads, 333 queries x 7, 5001 keys: 4 splits (608 workgroups, three to a unit) 83 us, 3 splits
// (456, two) 63 us, 5 splits (760, three) 73 us; 4 x 4 heads, 541 x 7 over 5238: 2 splits 177, none 152.
struct Splits {
  int n;
  bool pair;
  int64_t ns;
};
Splits pick_splits(const kvx_sdpa_args& a, int m_blocks, int num_tiles) {
  const int64_t base = (int64_t)a.B * a.Hkv * m_blocks, cus = num_cus();
  const bool plain = kv_is_plain(a.kv_dtype);
  int64_t tile_ns = a.D == 64 ? 840 : a.D == 128 ? 1130 : 2050;
  if (!plain) tile_ns = a.D == 256 ? 5500 : a.D == 64 ? 1700 : 2560;  // 256 rows a workgroup, codes to dequantise (at 256: 128 rows)
  const bool two = pairs(a.kv_dtype, a.D);
  const int64_t rows = (int64_t)a.B * a.Hq * a.q_len;
  Splits best = {1, false, INT64_MAX};
  for (int s = 1; s <= min(64, num_tiles); ++s) {
    const int tps = (num_tiles + s - 1) / s;
    if ((num_tiles + tps - 1) / tps != s) continue;
    const int64_t c = (base * s + cus - 1) / cus;
    // an odd workgroup after the pairs gains nothing and waits for one of them to end
    const int64_t partials = s * rows * (a.D * 4 + 8);
    const int64_t merge = s == 1 ? 0 : two ? 3400 + 30 * s + partials / 2000 : 2000 + partials / 4000;
    auto consider = [&](int64_t walk, bool pair) {
      if (walk + merge < best.ns) best = {s, pair, walk + merge};
    };
    if (!two) {
      consider(tps * tile_ns * c, false);
    } else {
      const int64_t side = a.D == 64 ? 3 : 2;  // side by side
      static const int64_t first[3] = {0, 100, 146}, after64[3] = {0, 113, 141}, after128[2] = {0, 106};
      const int64_t walk = c < side ? first[c] : a.D == 64 ? 195 * (c / 3) + after64[c % 3] : 148 * (c / 2) + after128[c % 2];
      consider(tps * tile_ns * walk / 100 + 200 * ((c + side - 1) / side), false);
      if (tps > 1) consider((tps + 1) / 2 * tile_ns * c * (a.D == 64 ? 150 : c == 1 ? 145 : 160) / 100 + 600 * c, true);
    }
  }
  return best;
}

// Splits of a causal first chunk (rows see the keys up to their own), by estimated time: tiles of a split, and whether a block of rows begins
// at the bounds of splits, for causal_job. Splits of all rows alike leave units idle: the jobs differ in length, those that see nothing still write and merge empty partials, and
// the best number of splits varies from size to size (8 heads of 128 over 2, 4096 tokens: 4 splits 68.5 us, 3 53.1, 2 60.7, one 79.4; 2048 tokens: 4
// 29.2, 3 31.1, 2 33.9, one 42.4). Here jobs without keys are not launched, a row merges the splits that it sees,
// and the jobs run in the order of their length (causal_job), so the walk takes the sum of the tiles that are seen and the jobs' begin and
// end, and a quarter of a split at the end; never less than one split, and more where two of them share a unit from the start. Calls of
// 8 heads over 2 of 4096 tokens 66.3 -> 56.7 us, of 2048 34.3 -> 27.5; 4 over 1, 8000 tokens 99.6 -> 82.2; 16 of 64 over 4, 3000 45.5 -> 40.6; 8 of
// 256 over 2, 3000 106.6 -> 74.4 (two splits of all rows alike are as good there, and at 4096 tokens three are better). Where the rows alone
// fill the device one split stays the best (32 over 8, 4096 tokens 133; two: 168). While a unit gets one job at most, splits of all rows alike can be
// shorter (a tile where bounds of blocks are two apart: one head of 256, 380 tokens 18.6 us in splits of two tiles, 15.5 in splits of one). A merge of
// their own counts as 4 us and 0.1 a split; as 2 us, the price in the score-sum launch (`combined`), splits were taken that one split beats: 24 heads of 256 over 8, 353 tokens 32.1 in three, 28.3 in one.
// Of 260 calls of 100 to 8000 tokens the splits chosen take 1.1 % longer than the best in the mean.
struct CausalSplits {
  int tiles;
  bool jobs;
};
CausalSplits causal_splits(const kvx_sdpa_args& a, int bm, int m_blocks, bool combined) {
  const int G = a.Hq / a.Hkv, tiles = (a.q_len + BN - 1) / BN;
  const int64_t groups = (int64_t)a.B * a.Hkv, cus = num_cus(), rows = groups * G * a.q_len;
  const int64_t tile_ns = a.D == 64 ? 700 : a.D == 128 ? 1130 : 2050, job_ns = 3000;
  const bool pairs = a.D <= 128;
  const int share = pairs ? 80 : 100;  // percent: two workgroups of a unit gain 20 %
  const int64_t seen = groups * m_blocks * (tiles + 1) / 2;
  int unit = 1;
  while (unit * BN * G % bm) unit *= 2;
  auto merge_ns = [&](int s) { return combined ? 2000 : 4000 + 100 * s; };
  CausalSplits best = {tiles, false};
  int64_t best_ns = INT64_MAX;
  auto consider = [&](int tps, bool jobs, int64_t walk, int64_t merge) {
    if (walk + merge >= best_ns) return;
    best_ns = walk + merge;
    best = {tps, jobs};
  };
  for (int s = 2; s <= min(16, tiles) && groups * m_blocks * s <= cus; ++s) {
    const int tps = (tiles + s - 1) / s;
    if ((tiles + tps - 1) / tps == s) consider(tps, false, tps * tile_ns + job_ns, merge_ns(s) + s * rows * (a.D * 4 + 8) / 4000);
  }
  for (int s = 1; s <= min(16, tiles); ++s) {
    const int tps = s == 1 ? tiles : ((tiles + s - 1) / s + unit - 1) / unit * unit;
    if (s > 1 && (tps >= tiles || (int64_t)m_blocks * (s + 1) / 2 + m_blocks > 65535)) break;  // (jobs are a grid's second dimension)
    const int64_t jobs = groups * m_blocks * (s + 1) / 2, one = tps * tile_ns + job_ns;
    const int64_t sum = (seen * tile_ns + jobs * job_ns) * share / 100 / cus;
    const int64_t alone = pairs && jobs > cus && jobs <= 2 * cus ? one * 115 / 100 : one;  // all at once, two to most units
    const int64_t walk = jobs <= cus ? one : std::max(alone, sum + (s == 1 ? 0 : one / 4));  // (max on the host is one of ints)
    const int64_t merge = s == 1 ? 0 : merge_ns(s) + rows * (s + 1) / 2 * (a.D * 4 + 8) / 4000;
    consider(tps, s > 1, walk, merge);
  }
  return best;
}

void fill_params(PrefillParams& p, const kvx_sdpa_args& a, bool combined = false) {
  common_params(p, a);
  const RowsPlan rows = rows_plan(a, combined);
  p.columns = rows.columns;
  const int bm = p.columns ? p.columns : 32 * nwaves(a.kv_dtype, a.D);
  p.m_blocks = (p.R + bm - 1) / bm;
  if (a.num_splits > 0) {
    p.num_splits = min(a.num_splits, p.num_tiles);
  } else if (p.columns) {
    p.num_splits = rows.splits;
  } else {
    const Splits s = pick_splits(a, p.m_blocks, p.num_tiles);
    p.num_splits = s.n;
    p.pair = s.pair;
  }
  p.tiles_per_split = (p.num_tiles + p.num_splits - 1) / p.num_splits;
  p.num_splits = (p.num_tiles + p.tiles_per_split - 1) / p.tiles_per_split;
  if (!a.token_positions && a.input_pos == 0 && a.q_len <= a.kv_len && kv_is_plain(a.kv_dtype) && a.num_splits <= 0 && !p.columns) {
    p.num_tiles = (a.q_len + BN - 1) / BN;  // nobody sees the keys behind
    const CausalSplits cs = causal_splits(a, bm, p.m_blocks, combined);
    p.tiles_per_split = cs.tiles;
    p.num_splits = (p.num_tiles + p.tiles_per_split - 1) / p.tiles_per_split;
    p.pair = 0;
    if (cs.jobs) p.period = p.tiles_per_split * BN * p.G / bm;
  }
}

size_t partial_bytes(const PrefillParams& p, int D) {
  if (p.num_splits <= 1) return 0;
  const size_t rows = (size_t)p.num_splits * p.B * p.Hkv * p.R;
  return rows * (size_t)D * 4 + rows * 2 * 4 * (p.pair ? 2 : 1);
}

MergeParams merge_params(const PrefillParams& p) {
  return {p.part_o, p.part_ml, p.o, p.lse, p.B, p.Hq, p.Hkv, p.G, p.q_len, p.R, p.num_splits, p.o_sb, p.o_sh, p.o_st,
          p.input_pos, p.tp ? 0 : p.tiles_per_split * BN, p.pair ? 2 : 1};
}

// `rest`: where the score-sum launch of `a` follows, what is left for it to combine (num_splits 1: nothing). `combined`: its kernel takes any splits
template <int D, int KV>
int launch_t(PrefillParams& p, const kvx_sdpa_args& a, hipStream_t st, MergeParams* rest, bool combined, const FirstWrite* write) {
  if (p.columns) {
    const int rc = launch_sdpa_rows(p, D, KV, st);
    if (rc != KVX_OK) return rc;
  } else {
    dim3 grid(p.B * p.Hkv, p.m_blocks, p.num_splits);
    if (p.period) {
      const int n = p.num_splits, last = p.m_blocks - (n - 1) * p.period;
      grid.y = (unsigned)(p.m_blocks + p.period * ((n - 1) * (n - 2) / 2) + last * (n - 1));
      grid.z = 1;
      if (combined) {  // the score-sum jobs read the maxima and sums of all splits of a row (its outputs are combined from those it sees)
        grid.y = (unsigned)p.m_blocks;
        grid.z = (unsigned)n;
        p.period = 0;
      }
    }
    bool general = true;
    if constexpr (kv_is_plain(KV)) {
      general = p.period == 0 && !write;
      if constexpr (D <= 128) {
        if (write && p.period) hipLaunchKernelGGL((sdpa_prefill_kernel<D, KV, true, false, true>), grid, dim3(64 * nwaves(KV, D)), 0, st, p, *write);
        if (write && !p.period) hipLaunchKernelGGL((sdpa_prefill_kernel<D, KV, false, false, true>), grid, dim3(64 * nwaves(KV, D)), 0, st, p, *write);
      }
      if (p.period && !write) hipLaunchKernelGGL((sdpa_prefill_kernel<D, KV, true, false>), grid, dim3(64 * nwaves(KV, D)), 0, st, p, NoWrite{});
    }
    if constexpr (pairs(KV, D)) {
      if (p.pair) {
        general = false;
        hipLaunchKernelGGL((sdpa_prefill_kernel<D, KV, false, true>), grid, dim3(2 * 64 * nwaves(KV, D)), 0, st, p, NoWrite{});
      }
    }
    if (general) hipLaunchKernelGGL((sdpa_prefill_kernel<D, KV, false, false>), grid, dim3(64 * nwaves(KV, D)), 0, st, p, NoWrite{});
    KVX_HIP(hipGetLastError());
  }
  const MergeParams m = merge_params(p);
  if (rest) {
    *rest = m;
    if (combined || (!p.period && score_sum_merges(a, m, false))) return KVX_OK;
    rest->num_splits = 1;
  }
  if (p.num_splits > 1) {
    auto merge = [&](auto sc_tag) {
      constexpr int SC = decltype(sc_tag)::value;
      hipLaunchKernelGGL((sdpa_prefill_merge_kernel<D, kv_elem_f16(KV), SC>), dim3((unsigned)merge_blocks(m, D, SC)), dim3(256), 0, st, m);
    };
    if (merge_wants_classes(m, D)) merge(std::integral_constant<int, merge_classes(D)>{});
    else merge(std::integral_constant<int, 1>{});
    KVX_HIP(hipGetLastError());
  }
  return KVX_OK;
}

}  // namespace

// Operands and sizes of a call, one split over all its keys.
void common_params(PrefillParams& p, const kvx_sdpa_args& a) {
  p.q = (const uint16_t*)a.q;
  p.k = a.k;
  p.v = a.v;
  p.k_scale = a.k_scale;
  p.k_zp = a.k_zp;
  p.v_scale = a.v_scale;
  p.v_zp = a.v_zp;
  p.tp = a.token_positions;
  p.o = (uint16_t*)a.o;
  p.lse = a.lse;
  p.B = a.B;
  p.Hq = a.Hq;
  p.Hkv = a.Hkv;
  p.G = a.Hq / a.Hkv;
  p.q_len = a.q_len;
  p.kv_len = a.kv_len;
  p.R = a.q_len * p.G;
  p.input_pos = a.input_pos;
  p.num_tiles = (a.kv_len + BN - 1) / BN;
  p.num_splits = 1;
  p.tiles_per_split = p.num_tiles;
  p.m_blocks = 0;
  p.period = 0;
  p.pair = 0;
  p.columns = 0;
  p.c = a.sm_scale * kLog2e;
  p.q_sb = a.q_stride_b; p.q_sh = a.q_stride_h; p.q_st = a.q_stride_t;
  p.k_sb = a.k_stride_b; p.k_sh = a.k_stride_h; p.k_st = a.k_stride_t;
  p.v_sb = a.v_stride_b; p.v_sh = a.v_stride_h; p.v_st = a.v_stride_t;
  p.o_sb = a.o_stride_b; p.o_sh = a.o_stride_h; p.o_st = a.o_stride_t;
  p.qs_sb = a.qs_stride_b; p.qs_sh = a.qs_stride_h;
  p.tp_sb = a.tp_stride_b; p.tp_sh = a.tp_stride_h;
  p.qs_vec = (((uintptr_t)a.k_scale | (uintptr_t)a.k_zp | (uintptr_t)a.v_scale | (uintptr_t)a.v_zp) & 15) == 0 && a.qs_stride_b % 4 == 0 && a.qs_stride_h % 4 == 0;
  p.tp_vec = ((uintptr_t)a.token_positions & 15) == 0 && a.tp_stride_b % 4 == 0 && a.tp_stride_h % 4 == 0;
  p.part_o = nullptr;
  p.part_ml = nullptr;
}

// Whether a call over a quantised store first dequantises the store into the workspace and then attends over plain rows.
// Every workgroup of the attention kernel walks the whole store (of its split) and the dequantising one pays its vector work
// each time, once per 256 rows; the copy pays it once, for one write and one more read of the 16-bit rows. Measured on
// 65536 x 8 rows of 128, 1024 x 4 queries: 1298 us against 75 + 1048. In units of 5 us there (8 x 32768 rows), a block of 256
// rows of the dequantising kernel takes 8, one of 128 of the plain kernel 3 and the copy 7: it pays from 1025 rows on, and
// below where 256-row blocks would be half empty. us, codes -> copy: 8 x 32768 8-bit rows of 128, 600 / 1024 / 1400 queries
// 133 -> 121, 168 -> 165, 261 -> 222; 16 x 6000 of 64, 1400 74 -> 66; 768 queries over the first 136 -> 137: not taken. Below 3 M
// values the copy's launch is what counts (8 x 1500 of 128, 600 queries 28.2 -> 28.9). At head size 256 the
// dequantising kernel runs 128 rows a workgroup out of its registers (4 x 4 heads, 541 x 7 queries over 5238: 890 us against
// 26 + 340), and the copy pays from the second workgroup on.
bool wants_copy(const kvx_sdpa_args& a) {
  if (kv_is_plain(a.kv_dtype) || (int64_t)a.B * a.Hkv > 65535) return false;  // pairs are a grid dimension of 16 bits
  const int64_t rows = (int64_t)a.q_len * (a.Hq / a.Hkv);
  if (a.D == 256) return rows > 128;
  if (rows >= 2048) return true;
  return (int64_t)a.B * a.Hkv * a.kv_len * a.D >= 3000000 && 8 * ((rows + 255) / 256) > 3 * ((rows + 127) / 128) + 7;
}
static size_t copy_bytes(const kvx_sdpa_args& a) { return ((size_t)2 * a.B * a.Hkv * a.kv_len * a.D * 2 + 255) / 256 * 256; }
// the block up to workspace_bytes: callers of the prefill calls may not have the rest
static kvx_sdpa_args prefill_block(const kvx_sdpa_args& a) {
  kvx_sdpa_args c{};
  memcpy(&c, &a, offsetof(kvx_sdpa_args, workspace_bytes) + sizeof(a.workspace_bytes));
  return c;
}
// the call on the dequantised rows at `rows` (K, then V, each (B, Hkv, kv_len, D))
static kvx_sdpa_args on_copy(const kvx_sdpa_args& a, void* rows) {
  kvx_sdpa_args c = prefill_block(a);
  c.kv_dtype = kv_elem_f16(a.kv_dtype) ? KVX_KV_F16 : KVX_KV_BF16;
  c.k = rows;
  c.v = (char*)rows + (size_t)a.B * a.Hkv * a.kv_len * a.D * 2;
  c.k_stride_t = c.v_stride_t = a.D;
  c.k_stride_h = c.v_stride_h = (int64_t)a.kv_len * a.D;
  c.k_stride_b = c.v_stride_b = (int64_t)a.Hkv * a.kv_len * a.D;
  return c;
}

int64_t prefill_ns(const kvx_sdpa_args& a) {
  const RowsPlan rows = rows_plan(a, score_sum_combines(a));
  const int bm = 32 * nwaves(a.kv_dtype, a.D);
  return rows.columns ? rows.ns : pick_splits(a, (int)(((int64_t)a.q_len * (a.Hq / a.Hkv) + bm - 1) / bm), (a.kv_len + BN - 1) / BN).ns;
}

int sdpa_prefill_block_rows(const kvx_sdpa_args& a, bool may_copy) {
  const kvx_sdpa_args c = may_copy && wants_copy(a) ? on_copy(a, nullptr) : prefill_block(a);
  PrefillParams p;
  fill_params(p, c);
  return p.columns ? p.columns : 32 * nwaves(c.kv_dtype, c.D);
}

kvx_prefill_plan sdpa_prefill_plan(const kvx_sdpa_args& a, bool may_copy) {
  kvx_prefill_plan plan{};
  plan.copied = may_copy && wants_copy(a);
  if (a.w && !plan.copied && rows_weights_plan(a, plan)) return plan;
  const kvx_sdpa_args c = plan.copied ? on_copy(a, nullptr) : prefill_block(a);
  plan.combined = a.w && score_sum_combines(a);
  PrefillParams p;
  fill_params(p, c, plan.combined);
  plan.block_rows = p.columns ? p.columns : 32 * nwaves(c.kv_dtype, c.D);
  plan.row_blocks = p.m_blocks;
  plan.splits = p.num_splits;
  plan.split_keys = p.tiles_per_split * BN;
  plan.teams = p.pair ? 2 : 1;
  plan.score_sum = a.w ? score_sum_kind(a) : KVX_SCORE_SUM_NONE;
  if (a.w && !p.period && score_sum_merges(a, merge_params(p), true)) plan.combined = 1;
  return plan;
}

size_t sdpa_prefill_workspace(const kvx_sdpa_args& a, bool may_copy) {
  PrefillParams p;
  const bool copy = may_copy && wants_copy(a);
  size_t partials = 0;
  bool merged = false;  // by the launches of the tiled score-sums
  for (const bool combined : {false, true}) {
    fill_params(p, copy ? on_copy(a, nullptr) : prefill_block(a), combined);
    partials = std::max(partials, partial_bytes(p, a.D));  // (max on the host is one of ints)
    if (!combined) merged = a.w && !p.period && score_sum_merges(a, merge_params(p), true);
  }
  // the score-sum pass that may follow on the same stream takes the place of the copy or of the partials, and where it combines those a place behind them
  const size_t sums = score_sum_workspace(a);
  const size_t own = copy ? copy_bytes(a) + partials : merged ? (partials + 15) / 16 * 16 + sums : partials;
  return std::max({own, sums, a.w ? rows_weights_workspace(a) : 0});  // (max on the host is one of ints)
}

// Whether the attention launch of a first chunk writes the chunk's rows too: the tiled kernel, for one team, over the rows that are written, where its workgroups
// are few: a write on its own runs at the memory's rate where it is long. us, two launches -> one: 253 tokens of 2 x 32 heads over 4 19.2 -> 14.7, 343 of 32 over 4
// 19.2 -> 16.6, 1163 of 32 over 8 35.7 -> 33.5, 2109 of 28 over 4 57.1 -> 55.5, 566 of 64 values, 2 x 16 heads over 8 16.7 -> 14.6; 1408 of 2 x 32 over 8 53.8 -> 53.1; but 1967
// of 16 over 8 45.4 -> 46.8, 4096 of 32 over 8 145.7 -> 146.3, 4214 166.1 -> 166.6, 8192 517 -> 518.
// And where a workgroup's share of the write, the rows of 128 / G tokens, is short, or there are workgroups enough that others' products run beside it: of up to three heads a KV
// head it is spread over the device by a launch of its own where blocks of rows a unit are fewer than its values / 12288, rows that are not quantised counting a third. Codes: 969 tokens of
// 8 heads over 8 (0.25 blocks a unit, 1.33 is the line) 21.8 -> 29.3, 304 of 4 x 8 over 8 17.7 -> 24.0, 516 of 16 over 8 (0.28, 0.67) 18.6 -> 20.5, 233 of 2 x 24 over 8 (0.38, 0.44) 15.7 -> 17.1, but
// 968 of 2 x 16 over 8 (1.0) 32.7 -> 32.4, 954 31.1 -> 29.8, 836 of 2 x 32 over 16 (1.75) 36.5 -> 33.5; plain 947 of 8 over 8 (0.25, 0.44) 20.4 -> 21.1, 419 of 4 x 8 over 8 (0.5) 18.3 -> 18.0.
// Over 303 such calls of 0.12 to 1.6 blocks a unit, 1 to 8 heads a KV head, the choice takes 0.04 % longer than the better of both in the mean,
// always one launch 1.9 %, always two 6 %.
static bool writes_first(const kvx_sdpa_args& a, const PrefillParams& p, const kvx_cache_write_args& w) {
  const int64_t blocks = (int64_t)p.B * p.Hkv * p.m_blocks, values = 128 * a.D / p.G / (kv_is_plain(w.kv_dtype) ? 3 : 1);
  return a.D <= 128 && kv_is_plain(a.kv_dtype) && !p.columns && !p.pair && !a.token_positions && a.input_pos == 0 && a.q_len == a.kv_len && w.B == a.B && w.Hkv == a.Hkv &&
         w.num == a.q_len && w.D == a.D && kv_elem_f16(w.kv_dtype) == kv_elem_f16(a.kv_dtype) && blocks <= 3 * num_cus() && (p.G > 3 || blocks * 12288 >= num_cus() * values) &&
         (p.G > 2 || a.q_len <= 1024);
}

bool sdpa_prefill_writes_first(const kvx_sdpa_args& a, const kvx_cache_write_args& w) {
  PrefillParams p;
  fill_params(p, prefill_block(a));
  return writes_first(a, p, w);
}

int launch_sdpa_prefill(const kvx_sdpa_args& a_in, bool may_copy, hipStream_t st, MergeParams* rest, const kvx_cache_write_args* first) {
  PrefillParams p;
  kvx_sdpa_args a = prefill_block(a_in);
  const bool combined = rest && score_sum_combines(a_in);
  if (may_copy && wants_copy(a)) {
    // a workspace too small for the copy (sized for another call, or by a caller that has no room): the fused form
    const kvx_sdpa_args c = on_copy(a, a.workspace);
    fill_params(p, c, combined);
    if (a.workspace && a.workspace_bytes >= copy_bytes(a) + partial_bytes(p, a.D)) {
      const int rc = launch_dequantize_kv(a, a.workspace, st);
      if (rc != KVX_OK) return rc;
      a = c;
      a.workspace = (char*)a_in.workspace + copy_bytes(a_in);
      a.workspace_bytes = a_in.workspace_bytes - copy_bytes(a_in);
    }
  }
  fill_params(p, a, combined);
  if (combined && (!a.workspace || a.workspace_bytes < partial_bytes(p, a.D))) fill_params(p, a);  // no room: the (fewer) splits of a call without weights
  const size_t need = partial_bytes(p, a.D);
  if (need) {
    KVX_REQUIRE(a.workspace && a.workspace_bytes >= need, KVX_ERR_WORKSPACE,
                "kvx_sdpa_prefill: workspace of %zu bytes needed, %zu given", need, a.workspace_bytes);
    const size_t rows = (size_t)p.num_splits * p.B * p.Hkv * p.R;
    p.part_o = (float*)a.workspace;
    p.part_ml = p.part_o + rows * (size_t)a.D;
  }
  FirstWrite fused;
  const FirstWrite* write = nullptr;
  if (first) {
    if (writes_first(a, p, *first)) {
      fused = {*first, (uint32_t)(first->cache_len - first->num)};
      write = &fused;
    } else {
      const int rc = launch_cache_write(*first, nullptr, st, first->cache_len > first->num);
      if (rc != KVX_OK) return rc;
    }
  }
#define KVX_PREFILL_CASE(KV) \
  case KV: return a.D == 256 ? launch_t<256, KV>(p, a_in, st, rest, combined, write) : a.D == 128 ? launch_t<128, KV>(p, a_in, st, rest, combined, write) : launch_t<64, KV>(p, a_in, st, rest, combined, write);
  if (a.D == 256 || a.D == 128 || a.D == 64) {
    switch (a.kv_dtype) {
      KVX_PREFILL_CASE(KVX_KV_BF16)
      KVX_PREFILL_CASE(KVX_KV_F16)
      KVX_PREFILL_CASE(KVX_KV_U8)
      KVX_PREFILL_CASE(KVX_KV_U4)
      KVX_PREFILL_CASE(KVX_KV_U8_F16)
      KVX_PREFILL_CASE(KVX_KV_U4_F16)
    }
  }
#undef KVX_PREFILL_CASE
  return set_error(KVX_ERR_UNSUPPORTED, "kvx_sdpa_prefill: head size %d not in {64, 128, 256}", a.D);
}

}  // namespace kvx
