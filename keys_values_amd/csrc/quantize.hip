// Affine 8-bit and 4-bit quantiser / dequantiser and the cache-slot write for gfx950 (HBM-bound byte work).
//
// Reference behaviour: keys_values/kvcache/quantize/pytorch.py:100-139,312-355 (quantise),
// :143-154,411-478 (dequantise); keys_values/kvcache/attn_weights.py:305-316,679-681 and
// keys_values/kvcache/buffers.py:498-519 (slot write).
//
// A row of D bf16 values is spread over D/8 adjacent lanes, 8 values (one 16-byte load) per lane,
// so a wavefront reads 1 KiB of contiguous input per load instruction and writes 512 contiguous
// bytes of codes. Row min and max are reduced with DPP moves inside the 16-lane row (no LDS).
#include "row_write.h"

namespace kvx {
namespace {

// Where the rows of a call lie: `n_outer` runs of `rows` rows each. A contiguous store is one run; a range of slots of a
// store is one run per (batch, head). A launch takes the runs along blockIdx.y.
struct RowRuns {
  uint16_t* x;
  int64_t x_row_stride, x_run_stride;  // elements
  uint8_t* codes;
  int64_t codes_run_stride;            // bytes; the rows of a run are adjacent
  float* scale;
  int32_t* zp;
  int64_t state_run_stride;            // elements
  int64_t rows;
  int n_outer;
};

template <int D, bool F16>
__global__ __launch_bounds__(NTHREADS) void quantize_rows_kernel(const RowRuns a) {
  const int64_t rows = a.rows, x_row_stride = a.x_row_stride;
  const uint16_t* __restrict__ x = a.x + blockIdx.y * a.x_run_stride;
  uint8_t* __restrict__ codes = a.codes + blockIdx.y * a.codes_run_stride;
  float* __restrict__ scale = a.scale + blockIdx.y * a.state_run_stride;
  int32_t* __restrict__ zp = a.zp + blockIdx.y * a.state_run_stride;
  constexpr int LPR = D / 8;
  constexpr int RPB = NTHREADS / LPR;  // rows per block per step
  const int col = threadIdx.x % LPR;
  const int64_t row0 = (int64_t)blockIdx.x * (RPB * ROWS_PER_THREAD) + threadIdx.x / LPR;
  u32x4_t raw[ROWS_PER_THREAD];
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD; ++i) {
    const int64_t r = row0 + (int64_t)i * RPB;
    raw[i] = r < rows ? __builtin_nontemporal_load((const u32x4_t*)(x + r * x_row_stride + col * 8)) : u32x4_t{0, 0, 0, 0};
  }
  u32x2_t c[ROWS_PER_THREAD];
  float s;
  int32_t z;
  quantize_rows_in_flight<LPR, 8, F16>(raw, c, s, z);  // executed by all lanes: the DPP exchanges need them
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD; ++i) {
    const int64_t r = row0 + (int64_t)i * RPB;
    if (r < rows) *(u32x2_t*)(codes + r * D + col * 8) = c[i];
  }
  // lane `col` of a row's first quad holds the state of row `col` of the four
  const int64_t r_mine = row0 + (int64_t)col * RPB;
  if (col < ROWS_PER_THREAD && r_mine < rows) {
    scale[r_mine] = s;
    zp[r_mine] = z;
  }
}

template <int D, bool F16>
__global__ __launch_bounds__(NTHREADS) void dequantize_rows_kernel(const RowRuns a) {
  const int64_t rows = a.rows, out_row_stride = a.x_row_stride;
  const uint8_t* __restrict__ codes = a.codes + blockIdx.y * a.codes_run_stride;
  const float* __restrict__ scale = a.scale + blockIdx.y * a.state_run_stride;
  const int32_t* __restrict__ zp = a.zp + blockIdx.y * a.state_run_stride;
  uint16_t* __restrict__ out = a.x + blockIdx.y * a.x_run_stride;
  constexpr int LPR = D / 8;
  constexpr int RPB = NTHREADS / LPR;
  const int col = threadIdx.x % LPR;
  const int64_t row0 = (int64_t)blockIdx.x * (RPB * ROWS_PER_THREAD) + threadIdx.x / LPR;
  u32x2_t c[ROWS_PER_THREAD];
  float s[ROWS_PER_THREAD];
  int32_t z[ROWS_PER_THREAD];
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD; ++i) {
    const int64_t r = row0 + (int64_t)i * RPB;
    const bool ok = r < rows;
    c[i] = ok ? *(const u32x2_t*)(codes + r * D + col * 8) : u32x2_t{0, 0};
    s[i] = ok ? scale[r] : 0.0f;
    z[i] = ok ? zp[r] : 0;
  }
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD; ++i) {
    const int64_t r = row0 + (int64_t)i * RPB;
    if (r >= rows) continue;
    *(u32x4_t*)(out + r * out_row_stride + col * 8) = dequant_words<F16>(c[i][0], c[i][1], z[i], s[i]);
  }
}

// ---- 4-bit rows -------------------------------------------------------------------------------

// Element d shares its byte with element d + D/2 (high nibble = first half of the row): the lanes of
// the first half fetch their partner's codes from the lane LPR/2 away and store 8 packed bytes.
template <int D, bool F16>
__global__ __launch_bounds__(NTHREADS) void quantize_rows4_kernel(const RowRuns a) {
  const int64_t rows = a.rows, x_row_stride = a.x_row_stride;
  const uint16_t* __restrict__ x = a.x + blockIdx.y * a.x_run_stride;
  uint8_t* __restrict__ codes = a.codes + blockIdx.y * a.codes_run_stride;
  float* __restrict__ scale = a.scale + blockIdx.y * a.state_run_stride;
  int32_t* __restrict__ zp = a.zp + blockIdx.y * a.state_run_stride;
  constexpr int LPR = D / 8;
  constexpr int RPB = NTHREADS / LPR;
  const int col = threadIdx.x % LPR;
  const int64_t row0 = (int64_t)blockIdx.x * (RPB * ROWS_PER_THREAD) + threadIdx.x / LPR;
  u32x4_t raw[ROWS_PER_THREAD];
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD; ++i) {
    const int64_t r = row0 + (int64_t)i * RPB;
    raw[i] = r < rows ? __builtin_nontemporal_load((const u32x4_t*)(x + r * x_row_stride + col * 8)) : u32x4_t{0, 0, 0, 0};
  }
  u32x2_t c[ROWS_PER_THREAD];
  float s;
  int32_t z;
  quantize_rows_in_flight<LPR, 4, F16>(raw, c, s, z);  // executed by all lanes: the reductions and the exchanges need them
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD; ++i) {
    const int64_t r = row0 + (int64_t)i * RPB;
    const uint32_t p0 = __shfl_xor(c[i][0], LPR / 2, 64), p1 = __shfl_xor(c[i][1], LPR / 2, 64);
    if (r < rows && col < LPR / 2) *(u32x2_t*)(codes + r * (D / 2) + col * 8) = u32x2_t{(c[i][0] << 4) | p0, (c[i][1] << 4) | p1};
  }
  const int64_t r_mine = row0 + (int64_t)col * RPB;
  if (col < ROWS_PER_THREAD && r_mine < rows) {
    scale[r_mine] = s;
    zp[r_mine] = z;
  }
}

// One lane per 8 packed bytes of ROWS_PER_THREAD rows: the high nibbles are elements col*8.., the low nibbles D/2 + col*8...
template <int D, bool F16>
__global__ __launch_bounds__(NTHREADS) void dequantize_rows4_kernel(const RowRuns a) {
  const int64_t rows = a.rows, out_row_stride = a.x_row_stride;
  const uint8_t* __restrict__ codes = a.codes + blockIdx.y * a.codes_run_stride;
  const float* __restrict__ scale = a.scale + blockIdx.y * a.state_run_stride;
  const int32_t* __restrict__ zp = a.zp + blockIdx.y * a.state_run_stride;
  uint16_t* __restrict__ out = a.x + blockIdx.y * a.x_run_stride;
  constexpr int LPR = D / 16;
  constexpr int RPB = NTHREADS / LPR;
  const int col = threadIdx.x % LPR;
  const int64_t row0 = (int64_t)blockIdx.x * (RPB * ROWS_PER_THREAD) + threadIdx.x / LPR;
  u32x2_t c[ROWS_PER_THREAD];
  float s[ROWS_PER_THREAD];
  int32_t z[ROWS_PER_THREAD];
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD; ++i) {
    const int64_t r = row0 + (int64_t)i * RPB;
    const bool ok = r < rows;
    c[i] = ok ? *(const u32x2_t*)(codes + r * (D / 2) + col * 8) : u32x2_t{0, 0};
    s[i] = ok ? scale[r] : 0.0f;
    z[i] = ok ? zp[r] : 0;
  }
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD; ++i) {
    const int64_t r = row0 + (int64_t)i * RPB;
    if (r >= rows) continue;
    u32x4_t hi, lo;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t w = c[i][e >> 1] >> ((e & 1) * 16);
      hi[e] = dequant_pair<F16>((w >> 4) & 0xf, (w >> 12) & 0xf, z[i], s[i]);
      lo[e] = dequant_pair<F16>(w & 0xf, (w >> 8) & 0xf, z[i], s[i]);
    }
    *(u32x4_t*)(out + r * out_row_stride + col * 8) = hi;
    *(u32x4_t*)(out + r * out_row_stride + D / 2 + col * 8) = lo;
  }
}

// K (blockIdx.z = 0) and V (1) of an attention call's quantised store to dense rows: a (batch, KV head) pair per blockIdx.y and blocks of its rows along
// blockIdx.x, or the other way round (by_pair). A lane owns 8 values of ROWS_PER_THREAD rows, as above; the codes' rows lie wherever the strides say.
template <int D, int KV>
__global__ __launch_bounds__(NTHREADS) void dequantize_kv_kernel(const kvx_sdpa_args a, uint16_t* __restrict__ out, const bool by_pair) {
  constexpr bool U4 = kv_is_u4(KV), F16 = kv_elem_f16(KV);
  constexpr int LPR = U4 ? D / 16 : D / 8;  // lanes per row: 8 bytes of codes each
  constexpr int RPB = NTHREADS / LPR;
  const bool is_v = blockIdx.z != 0;
  const int pair = by_pair ? blockIdx.x : blockIdx.y, at = by_pair ? blockIdx.y : blockIdx.x;
  const int b = pair / a.Hkv, h = pair % a.Hkv;
  const int64_t sb = is_v ? a.v_stride_b : a.k_stride_b, sh = is_v ? a.v_stride_h : a.k_stride_h, stt = is_v ? a.v_stride_t : a.k_stride_t;
  const uint8_t* __restrict__ codes = (const uint8_t*)(is_v ? a.v : a.k) + b * sb + h * sh;
  const int64_t so = b * a.qs_stride_b + h * a.qs_stride_h;
  const float* __restrict__ scale = (is_v ? a.v_scale : a.k_scale) + so;
  const int32_t* __restrict__ zp = (is_v ? a.v_zp : a.k_zp) + so;
  uint16_t* __restrict__ o = out + ((int64_t)blockIdx.z * a.B * a.Hkv + pair) * a.kv_len * D;
  const int col = threadIdx.x % LPR;
  const int row0 = at * (RPB * ROWS_PER_THREAD) + threadIdx.x / LPR;
  u32x2_t c[ROWS_PER_THREAD];
  float s[ROWS_PER_THREAD];
  int32_t z[ROWS_PER_THREAD];
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD; ++i) {
    const int r = min(row0 + i * RPB, a.kv_len - 1);
    c[i] = *(const u32x2_t*)(codes + r * stt + col * 8);
    s[i] = scale[r];
    z[i] = zp[r];
  }
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD; ++i) {
    const int r = row0 + i * RPB;
    if (r >= a.kv_len) continue;
    uint16_t* w = o + (int64_t)r * D + col * 8;
    if constexpr (U4) {
      const u32x2_t hi = u4_codes(c[i], 4), lo = u4_codes(c[i], 0);
      *(u32x4_t*)w = dequant_words<F16>(hi[0], hi[1], z[i], s[i]);
      *(u32x4_t*)(w + D / 2) = dequant_words<F16>(lo[0], lo[1], z[i], s[i]);
    } else {
      *(u32x4_t*)w = dequant_words<F16>(c[i][0], c[i][1], z[i], s[i]);
    }
  }
}

// ---- general blocks (several segments per block, 8 or 4 bits) -------------------------------------------------------
//
// A block of n chunks of 8 values (n is even: D is a multiple of 16) is held by LPB lanes, lane l taking the chunk pairs
// (l + LPB i, l + LPB i + n / 2), i < NP: the two halves of the block are what shares the bytes of the 4-bit store, and
// two 16-byte loads a pair keep enough bytes in flight. LPB is the power of two from 8 to 64 that n / 2 needs, so short
// blocks share a wavefront; longer ones take up to NP = 8 pairs a lane. The values stay in registers between the
// extremes and the codes: HBM sees every byte once.

template <bool F16>
__device__ __forceinline__ u32x2_t codes_of_chunk(u32x4_t raw, float inv, float zf, float qmax) {
  u32x2_t out;
#pragma unroll
  for (int h = 0; h < 2; ++h)
    out[h] = quant_code(elem_lo<F16>(raw[2 * h]), inv, zf, qmax) | (quant_code(elem_hi<F16>(raw[2 * h]), inv, zf, qmax) << 8) |
             (quant_code(elem_lo<F16>(raw[2 * h + 1]), inv, zf, qmax) << 16) | (quant_code(elem_hi<F16>(raw[2 * h + 1]), inv, zf, qmax) << 24);
  return out;
}

// Addresses of this lane's chunks; cps = chunks per segment, magic = ceil(2^21 / cps): c / cps == c magic >> 21 for c < 1024.
template <int LPB, int NP>
struct BlockLane {
  bool live;
  int64_t outer, inner;
  uint16_t* base;
  int half, cps, sub;
  uint32_t magic;
  int64_t seg;
  __device__ __forceinline__ BlockLane(const kvx_block_quant_args& a, uint32_t magic_) : magic(magic_) {
    const int64_t blk = ((int64_t)blockIdx.x * NTHREADS + threadIdx.x) / LPB;
    live = blk < (int64_t)a.n_outer * a.n_inner;
    const int64_t b = live ? blk : 0;
    outer = b / a.n_inner;
    inner = b % a.n_inner;
    base = (uint16_t*)a.x + outer * a.x_stride_outer + inner * a.x_stride_inner;
    cps = a.D / 8;
    half = a.nseg * cps / 2;
    sub = threadIdx.x % LPB;
    seg = a.x_stride_seg;
  }
  __device__ __forceinline__ int pair(int i) const { return sub + LPB * i; }
  __device__ __forceinline__ u32x4_t* chunk(int c) const {
    const int s = (int)(((uint32_t)c * magic) >> 21);
    return (u32x4_t*)(base + s * seg + (c - s * cps) * 8);
  }
};

template <int BITS, bool F16, int LPB, int NP>
__global__ __launch_bounds__(NTHREADS) void quantize_blocks_kernel(const kvx_block_quant_args a, const uint32_t magic) {
  const BlockLane<LPB, NP> bl(a, magic);
  u32x4_t raw[NP][2];
  float mn = INFINITY, mx = -INFINITY;
  bool bad = false;
#pragma unroll
  for (int i = 0; i < NP; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      raw[i][h] = bl.live && bl.pair(i) < bl.half ? __builtin_nontemporal_load(bl.chunk(bl.pair(i) + h * bl.half)) : u32x4_t{0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (bl.pair(i) < bl.half) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float lo = elem_lo<F16>(raw[i][h][e]), hi = elem_hi<F16>(raw[i][h][e]);
          mn = fminf(mn, fminf(lo, hi));
          mx = fmaxf(mx, fmaxf(lo, hi));
          bad |= __builtin_isunordered(lo, hi);
        }
    }
#pragma unroll
  for (int off = LPB / 2; off >= 1; off >>= 1) {
    mn = fminf(mn, __shfl_xor(mn, off, 64));
    mx = fmaxf(mx, __shfl_xor(mx, off, 64));
  }
  if (row_any<LPB>(bad)) mn = mx = __builtin_nanf("");  // as torch.aminmax: a NaN in the block is the block's extreme
  if (!bl.live) return;
  constexpr float qmax = BITS == 8 ? 255.0f : 15.0f;
  float s;
  int32_t z;
  quant_params(mn, mx, s, z, qmax);
  const float inv = 1.0f / s, zf = (float)z;
  uint8_t* out = a.codes + bl.outer * a.codes_stride_outer + bl.inner * ((int64_t)bl.half * 2 * BITS);  // 8 values a chunk, BITS / 8 bytes each
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (bl.pair(i) < bl.half) {
      const u32x2_t c0 = codes_of_chunk<F16>(raw[i][0], inv, zf, qmax), c1 = codes_of_chunk<F16>(raw[i][1], inv, zf, qmax);
      if constexpr (BITS == 8) {
        *(u32x2_t*)(out + bl.pair(i) * 8) = c0;
        *(u32x2_t*)(out + (bl.pair(i) + bl.half) * 8) = c1;
      } else {
        *(u32x2_t*)(out + bl.pair(i) * 8) = u32x2_t{(c0[0] << 4) | c1[0], (c0[1] << 4) | c1[1]};
      }
    }
  if (bl.sub == 0) {
    a.scale[bl.outer * a.state_stride_outer + bl.inner] = s;
    a.zp[bl.outer * a.state_stride_outer + bl.inner] = z;
  }
}

template <int BITS, bool F16, int LPB, int NP>
__global__ __launch_bounds__(NTHREADS) void dequantize_blocks_kernel(const kvx_block_quant_args a, const uint32_t magic) {
  const BlockLane<LPB, NP> bl(a, magic);
  if (!bl.live) return;
  const float s = a.scale[bl.outer * a.state_stride_outer + bl.inner];
  const int32_t z = a.zp[bl.outer * a.state_stride_outer + bl.inner];
  const uint8_t* in = a.codes + bl.outer * a.codes_stride_outer + bl.inner * ((int64_t)bl.half * 2 * BITS);
  u32x2_t c[NP][2];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const bool ok = bl.pair(i) < bl.half;
    c[i][0] = ok ? *(const u32x2_t*)(in + bl.pair(i) * 8) : u32x2_t{0, 0};
    if constexpr (BITS == 8) c[i][1] = ok ? *(const u32x2_t*)(in + (bl.pair(i) + bl.half) * 8) : u32x2_t{0, 0};
  }
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (bl.pair(i) < bl.half) {
      u32x2_t c0 = c[i][0], c1 = c[i][1];
      if constexpr (BITS == 4) {
        c1 = u4_codes(c0, 0);
        c0 = u4_codes(c0, 4);
      }
      *bl.chunk(bl.pair(i)) = dequant_words<F16>(c0[0], c0[1], z, s);
      *bl.chunk(bl.pair(i) + bl.half) = dequant_words<F16>(c1[0], c1[1], z, s);
    }
}

constexpr int CLEARED = 4;  // slots a thread clears

// One lane per 8 elements of one job (b, h, j), for K and V. Without a ring move job j writes new
// token j into index[b,h,j]. With one (j < grace_num) the lanes of the job first carry ring slot
// grace_slots[j] over to index[b,h,j], then write new token num - grace_num + j into the ring slot:
// the read and the write of that slot are issued by the same wavefront, in this order, and the
// read's data is consumed before the write is issued.
template <int D, int KV>
__global__ __launch_bounds__(NTHREADS) void cache_write_kernel(const kvx_cache_write_args a, const DecodeCounters clear, const uint32_t jobs, const uint32_t rest) {
  constexpr bool U8 = !kv_is_plain(KV);  // a quantised store: codes + row state
  constexpr bool U4 = kv_is_u4(KV);       // two codes per byte: only the lanes of the first half of a row store
  constexpr bool F16 = kv_elem_f16(KV);   // the rows are float16
  constexpr int LPR = D / 8;
  // workgroups behind the jobs': `rest` slots of every row, behind the written ones, are cleared
  const uint32_t job_blocks = (jobs + NTHREADS / LPR - 1) / (NTHREADS / LPR);
  if (blockIdx.x >= job_blocks) {
    const uint32_t total = (uint32_t)(a.B * a.Hkv) * rest;
#pragma unroll
    for (int i = 0; i < CLEARED; ++i) {
      const uint32_t at = ((blockIdx.x - job_blocks) * CLEARED + i) * NTHREADS + threadIdx.x;
      if (at >= total) return;
      const uint32_t row = at / rest;
      const int64_t to = row / a.Hkv * a.sc_stride_b + row % a.Hkv * a.sc_stride_h + a.num + (at - row * rest);
      if (a.scores) a.scores[to] = 0.0f;
      if (a.v_norm) a.v_norm[to] = 0.0f;
      if (a.q_errors) a.q_errors[to] = 0.0f;
    }
    return;
  }
  const int64_t gid = (int64_t)blockIdx.x * NTHREADS + threadIdx.x;
  if (clear.rows) {  // one line per (batch, KV head) row: there are at least as many lanes (LPR of them a job)
    clear_counters(clear, gid, (int64_t)gridDim.x * NTHREADS, (int64_t)a.B * a.Hkv);
    if (gid == 0 && clear.scratch_splits) *clear.scratch_splits = 0u;
  }
  const int col = threadIdx.x % LPR;
  const uint32_t rid = blockIdx.x * (NTHREADS / LPR) + threadIdx.x / LPR;
  const bool live = rid < jobs;
  const uint32_t ridc = live ? rid : 0, pair = ridc / (uint32_t)a.num;
  const int j = (int)(ridc - pair * a.num);
  const int b = (int)(pair / (uint32_t)a.Hkv), hh = (int)(pair - b * a.Hkv);
  const int slot = a.index[b * a.index_stride_b + hh * a.index_stride_h + j];
  const bool moves = j < a.grace_num;
  const int ring = moves ? a.grace_slots[j] : -1;
  const int src = moves ? a.num - a.grace_num + j : j - a.grace_num;  // new token this job stores
  // a bad index is dropped, never written out of bounds
  const bool ok = live && slot >= 0 && slot < a.cache_len && (!moves || (ring >= 0 && ring < a.cache_len && ring != slot));
  const int wslot = moves ? ring : slot;  // where the new token goes
  const uint16_t* ks = (const uint16_t*)a.key + b * a.key_stride_b + hh * a.key_stride_h + (int64_t)src * a.key_stride_t + col * 8;
  const uint16_t* vs = (const uint16_t*)a.value + b * a.value_stride_b + hh * a.value_stride_h + (int64_t)src * a.value_stride_t + col * 8;
  const u32x4_t kr = live ? *(const u32x4_t*)ks : u32x4_t{0, 0, 0, 0};
  const u32x4_t vr = live ? *(const u32x4_t*)vs : u32x4_t{0, 0, 0, 0};
  const int64_t tp_row = b * a.tp_stride_b + hh * a.tp_stride_h;
  const int64_t sc_row = b * a.sc_stride_b + hh * a.sc_stride_h;
  const int64_t qs_row = b * a.qs_stride_b + hh * a.qs_stride_h;
  constexpr int ES = U8 ? 1 : 2;  // bytes per cache element
  const int ccol = U4 ? col % (LPR / 2) : col;
  uint8_t* kc_row = (uint8_t*)a.k_cache + (b * a.kc_stride_b + hh * a.kc_stride_h) * ES + ccol * 8 * ES;
  uint8_t* vc_row = (uint8_t*)a.v_cache + (b * a.vc_stride_b + hh * a.vc_stride_h) * ES + ccol * 8 * ES;

  auto put = [&](const u32x4_t& krow, const u32x4_t& vrow, int target, bool doit, bool want_err) {
    return put_rows<D, KV>(a, kc_row, vc_row, qs_row, col, krow, vrow, target, doit, want_err);
  };

  if (a.grace_num > 0) {  // uniform over the launch
    const bool mv = ok && moves;
    if constexpr (!U8) {
      if (mv) {
        *(u32x4_t*)(kc_row + (int64_t)slot * a.kc_stride_t * ES) = *(const u32x4_t*)(kc_row + (int64_t)ring * a.kc_stride_t * ES);
        *(u32x4_t*)(vc_row + (int64_t)slot * a.vc_stride_t * ES) = *(const u32x4_t*)(vc_row + (int64_t)ring * a.vc_stride_t * ES);
      }
    } else {
      // The moved row is written like any other: its dequantised values are quantised again
      // (keys_values/kvcache/attn_weights.py:578-590 reads the ring rows from the dequantised buffer
      // and hands them to the same write as the new rows), which is not the identity on the codes.
      u32x4_t krow = {0, 0, 0, 0}, vrow = {0, 0, 0, 0};
      if (mv) {
        u32x2_t kq = *(const u32x2_t*)(kc_row + (int64_t)ring * a.kc_stride_t);
        u32x2_t vq = *(const u32x2_t*)(vc_row + (int64_t)ring * a.vc_stride_t);
        if constexpr (U4) {
          kq = u4_codes(kq, col < LPR / 2 ? 4 : 0);
          vq = u4_codes(vq, col < LPR / 2 ? 4 : 0);
        }
        krow = dequant_words<F16>(kq[0], kq[1], a.k_zp[qs_row + ring], a.k_scale[qs_row + ring]);
        vrow = dequant_words<F16>(vq[0], vq[1], a.v_zp[qs_row + ring], a.v_scale[qs_row + ring]);
      }
      put(krow, vrow, slot, mv, false);
    }
    if (mv && col == 0) {
      if (a.token_pos) a.token_pos[tp_row + slot] = a.input_pos - a.grace_period + j;
      if (a.scores) a.scores[sc_row + slot] = a.scores[sc_row + ring];
      if (a.v_norm) a.v_norm[sc_row + slot] = a.v_norm[sc_row + ring];
      if (a.q_errors) a.q_errors[sc_row + slot] = a.q_errors[sc_row + ring];
    }
  }

  float qerr = 0.0f;
  if constexpr (!U8) {
    if (ok) {
      *(u32x4_t*)(kc_row + (int64_t)wslot * a.kc_stride_t * ES) = kr;
      *(u32x4_t*)(vc_row + (int64_t)wslot * a.vc_stride_t * ES) = vr;
    }
  } else {
    qerr = put(kr, vr, wslot, ok, a.q_errors != nullptr);
  }
  float vnorm = 0.0f;
  if (a.v_norm) vnorm = row_norm<LPR, F16>(vr);  // uniform branch: every lane takes part in the reduction
  if (live && col == 0 && a.replay_log) {  // the slot as consumed, valid or not: the log mirrors index
    const int64_t lp = a.log_pos + j;
    a.replay_log[(lp / a.log_blocksize) * a.log_stride_block + b * a.log_stride_b + hh * a.log_stride_h + lp % a.log_blocksize] =
        (uint32_t)slot;
  }
  if (ok && col == 0) {
    if (a.token_pos) a.token_pos[tp_row + wslot] = a.input_pos + src;
    if (a.scores) a.scores[sc_row + wslot] = 0.0f;
    if (a.v_norm) a.v_norm[sc_row + wslot] = vnorm;
    if (a.q_errors) a.q_errors[sc_row + wslot] = qerr;
  }
}

}  // namespace

// D in {64, 128, 256}, bits in {8, 4}, f16: the rows are float16 (else bfloat16)
template <int D, bool F16>
int launch_rows_t(const RowRuns& a, int bits, bool quantize, hipStream_t st) {
  const int lpr = bits == 4 && !quantize ? D / 16 : D / 8;
  const int rpb = (NTHREADS / lpr) * ROWS_PER_THREAD;
  RowRuns r = a;
  for (int done = 0; done < a.n_outer; done += 65535) {  // runs along a grid dimension of 16 bits
    const dim3 grid((unsigned)((a.rows + rpb - 1) / rpb), (unsigned)min(a.n_outer - done, 65535));
    if (quantize && bits == 8) hipLaunchKernelGGL((quantize_rows_kernel<D, F16>), grid, dim3(NTHREADS), 0, st, r);
    else if (quantize) hipLaunchKernelGGL((quantize_rows4_kernel<D, F16>), grid, dim3(NTHREADS), 0, st, r);
    else if (bits == 8) hipLaunchKernelGGL((dequantize_rows_kernel<D, F16>), grid, dim3(NTHREADS), 0, st, r);
    else hipLaunchKernelGGL((dequantize_rows4_kernel<D, F16>), grid, dim3(NTHREADS), 0, st, r);
    KVX_HIP(hipGetLastError());
    r.x += 65535 * a.x_run_stride;
    r.codes += 65535 * a.codes_run_stride;
    r.scale += 65535 * a.state_run_stride;
    r.zp += 65535 * a.state_run_stride;
  }
  return KVX_OK;
}

static int launch_rows(const RowRuns& a, int D, int bits, bool f16, bool quantize, hipStream_t st) {
  if (a.rows == 0 || a.n_outer == 0) return KVX_OK;
  if (D == 256) return f16 ? launch_rows_t<256, true>(a, bits, quantize, st) : launch_rows_t<256, false>(a, bits, quantize, st);
  if (D == 128) return f16 ? launch_rows_t<128, true>(a, bits, quantize, st) : launch_rows_t<128, false>(a, bits, quantize, st);
  return f16 ? launch_rows_t<64, true>(a, bits, quantize, st) : launch_rows_t<64, false>(a, bits, quantize, st);
}

int launch_quantize_rows(const void* x, int64_t x_row_stride, int64_t rows, int D, int bits, bool f16, uint8_t* codes, float* scale,
                         int32_t* zp, hipStream_t st) {
  return launch_rows(RowRuns{(uint16_t*)x, x_row_stride, 0, codes, 0, scale, zp, 0, rows, 1}, D, bits, f16, true, st);
}

int launch_dequantize_rows(const uint8_t* codes, const float* scale, const int32_t* zp, int64_t rows, int D, int bits, bool f16,
                           void* out, int64_t out_row_stride, hipStream_t st) {
  return launch_rows(RowRuns{(uint16_t*)out, out_row_stride, 0, (uint8_t*)codes, 0, (float*)scale, (int32_t*)zp, 0, rows, 1}, D, bits, f16, false, st);
}

// While the 16-bit rows of K and V, 32 MB at 8 M values each, fit the L2 caches of the eight dies, pairs are the fastest index: the rows are written on the die whose
// attention workgroups read them. Beyond, no reader finds them there, and in the rows' order the writes run the faster. Rows' order against pairs' (us;
// attention of 512 queries of four heads behind it): calls over 16 x 1500 rows of 128 70.9, 68.3; 16 x 2000 of 64 92.0, 88.6; 8 x 5000 and 8 x 7000 alike; copies
// of 8 x 16384 15.8, 16.2; 8 x 32768 31.9, 33.7; 8 x 65536 60.2, 63.6, of 4-bit codes 52.6, 55.4.
constexpr int64_t COPY_BY_PAIR = 8ll << 20;
template <int D>
int launch_dequantize_kv_d(const kvx_sdpa_args& a, void* out, hipStream_t st) {
  const int lpr = kv_is_u4(a.kv_dtype) ? D / 16 : D / 8, rpb = NTHREADS / lpr * ROWS_PER_THREAD;
  const unsigned pairs = (unsigned)(a.B * a.Hkv), blocks = (unsigned)(a.kv_len / rpb + (a.kv_len % rpb != 0));
  KVX_REQUIRE(blocks < (1u << 24), KVX_ERR_UNSUPPORTED, "dequantised copy: %u blocks of rows, must be below 2^24", blocks);  // a dimension's threads are counted in 32 bits
  const bool by_pair = (int64_t)pairs * a.kv_len * D <= COPY_BY_PAIR;
  const dim3 grid(by_pair ? pairs : blocks, by_pair ? blocks : pairs, 2);
  switch (a.kv_dtype) {
    case KVX_KV_U8: hipLaunchKernelGGL((dequantize_kv_kernel<D, KVX_KV_U8>), grid, dim3(NTHREADS), 0, st, a, (uint16_t*)out, by_pair); break;
    case KVX_KV_U4: hipLaunchKernelGGL((dequantize_kv_kernel<D, KVX_KV_U4>), grid, dim3(NTHREADS), 0, st, a, (uint16_t*)out, by_pair); break;
    case KVX_KV_U8_F16: hipLaunchKernelGGL((dequantize_kv_kernel<D, KVX_KV_U8_F16>), grid, dim3(NTHREADS), 0, st, a, (uint16_t*)out, by_pair); break;
    default: hipLaunchKernelGGL((dequantize_kv_kernel<D, KVX_KV_U4_F16>), grid, dim3(NTHREADS), 0, st, a, (uint16_t*)out, by_pair); break;
  }
  KVX_HIP(hipGetLastError());
  return KVX_OK;
}

int launch_dequantize_kv(const kvx_sdpa_args& a, void* out, hipStream_t st) {
  return a.D == 256 ? launch_dequantize_kv_d<256>(a, out, st) : a.D == 128 ? launch_dequantize_kv_d<128>(a, out, st) : launch_dequantize_kv_d<64>(a, out, st);
}

template <int BITS, bool F16, int LPB, int NP>
int launch_blocks_t(const kvx_block_quant_args& a, bool quantize, hipStream_t st) {
  const int64_t lanes = (int64_t)a.n_outer * a.n_inner * LPB;
  const unsigned grid = (unsigned)((lanes + NTHREADS - 1) / NTHREADS);
  const uint32_t cps = (uint32_t)a.D / 8, magic = ((1u << 21) + cps - 1) / cps;
  if (quantize) hipLaunchKernelGGL((quantize_blocks_kernel<BITS, F16, LPB, NP>), dim3(grid), dim3(NTHREADS), 0, st, a, magic);
  else hipLaunchKernelGGL((dequantize_blocks_kernel<BITS, F16, LPB, NP>), dim3(grid), dim3(NTHREADS), 0, st, a, magic);
  KVX_HIP(hipGetLastError());
  return KVX_OK;
}

template <int BITS, bool F16>
int launch_blocks_bits(const kvx_block_quant_args& a, bool quantize, hipStream_t st) {
  const int half = a.nseg * a.D / 16;  // chunk pairs of a block, 1 .. 512
  if (half <= 8) return launch_blocks_t<BITS, F16, 8, 1>(a, quantize, st);
  if (half <= 16) return launch_blocks_t<BITS, F16, 16, 1>(a, quantize, st);
  if (half <= 32) return launch_blocks_t<BITS, F16, 32, 1>(a, quantize, st);
  if (half <= 64) return launch_blocks_t<BITS, F16, 64, 1>(a, quantize, st);
  if (half <= 128) return launch_blocks_t<BITS, F16, 64, 2>(a, quantize, st);
  if (half <= 256) return launch_blocks_t<BITS, F16, 64, 4>(a, quantize, st);
  return launch_blocks_t<BITS, F16, 64, 8>(a, quantize, st);
}

// One segment of 64, 128 or 256 values is a row: the row kernels (four rows in flight a lane, the state's arithmetic
// shared between them) serve a range of slots as one run per (batch, head), or as a single run where the runs are adjacent.
// Measured, one (1, 8, 65536, 128) tensor of 8-bit codes to rows: 99 us with a wavefront per row, 33 us this way.
static int launch_blocks(const kvx_block_quant_args& a, bool quantize, hipStream_t st) {
  if (a.n_outer == 0 || a.n_inner == 0) return KVX_OK;
  const bool f16 = a.elem_dtype == KVX_KV_F16;
  const int64_t code_bytes = (int64_t)a.D * a.bits / 8;
  if (a.nseg == 1 && (a.D == 64 || a.D == 128 || a.D == 256)) {
    RowRuns r{(uint16_t*)a.x, a.x_stride_inner, a.x_stride_outer, a.codes, a.codes_stride_outer, a.scale, a.zp, a.state_stride_outer, a.n_inner, a.n_outer};
    if (r.x_run_stride == r.rows * r.x_row_stride && r.codes_run_stride == r.rows * code_bytes && r.state_run_stride == r.rows) {
      r.rows *= r.n_outer;
      r.n_outer = 1;
    }
    return launch_rows(r, a.D, a.bits, f16, quantize, st);
  }
  if (a.bits == 8) return f16 ? launch_blocks_bits<8, true>(a, quantize, st) : launch_blocks_bits<8, false>(a, quantize, st);
  return f16 ? launch_blocks_bits<4, true>(a, quantize, st) : launch_blocks_bits<4, false>(a, quantize, st);
}

int launch_quantize_blocks(const kvx_block_quant_args& a, hipStream_t st) { return launch_blocks(a, true, st); }
int launch_dequantize_blocks(const kvx_block_quant_args& a, hipStream_t st) { return launch_blocks(a, false, st); }

template <int D>
int launch_cache_write_d(const kvx_cache_write_args& a, const DecodeCounters& clear, unsigned grid, uint32_t jobs, uint32_t rest, hipStream_t st) {
  switch (a.kv_dtype) {
    case KVX_KV_F16: hipLaunchKernelGGL((cache_write_kernel<D, KVX_KV_F16>), dim3(grid), dim3(NTHREADS), 0, st, a, clear, jobs, rest); break;
    case KVX_KV_BF16: hipLaunchKernelGGL((cache_write_kernel<D, KVX_KV_BF16>), dim3(grid), dim3(NTHREADS), 0, st, a, clear, jobs, rest); break;
    case KVX_KV_U4: hipLaunchKernelGGL((cache_write_kernel<D, KVX_KV_U4>), dim3(grid), dim3(NTHREADS), 0, st, a, clear, jobs, rest); break;
    case KVX_KV_U8: hipLaunchKernelGGL((cache_write_kernel<D, KVX_KV_U8>), dim3(grid), dim3(NTHREADS), 0, st, a, clear, jobs, rest); break;
    case KVX_KV_U4_F16: hipLaunchKernelGGL((cache_write_kernel<D, KVX_KV_U4_F16>), dim3(grid), dim3(NTHREADS), 0, st, a, clear, jobs, rest); break;
    default: hipLaunchKernelGGL((cache_write_kernel<D, KVX_KV_U8_F16>), dim3(grid), dim3(NTHREADS), 0, st, a, clear, jobs, rest); break;
  }
  KVX_HIP(hipGetLastError());
  return KVX_OK;
}

// Workgroups for the rows, and behind them for the `rest` slots of each (batch, KV head) row that a first chunk leaves empty
static uint32_t rest_of(const kvx_cache_write_args& a, bool first) { return first ? (uint32_t)(a.cache_len - a.num) : 0; }
int64_t cache_write_workgroups(const kvx_cache_write_args& a, bool first) {
  const int64_t pairs = (int64_t)a.B * a.Hkv;
  return (pairs * a.num * (a.D / 8) + NTHREADS - 1) / NTHREADS + (pairs * rest_of(a, first) + CLEARED * NTHREADS - 1) / (CLEARED * NTHREADS);
}

int launch_cache_write(const kvx_cache_write_args& a, const DecodeCounters* clear, hipStream_t st, bool first) {
  const DecodeCounters none{}, &c = clear ? *clear : none;
  if ((int64_t)a.B * a.Hkv * a.num * (a.D / 8) == 0) return KVX_OK;
  // A launch each for scores, norms and errors was 2 to 5 us, the most of a short first chunk (us, calls in a row: 90 tokens of 24 heads, 512 slots 19.1 -> 15.0; 384,
  // 2803 slots, norms and errors 29.0 -> 18.3; 8192 of 16384 slots 515.5 -> 511.9).
  const uint32_t rest = rest_of(a, first);
  const unsigned grid = (unsigned)cache_write_workgroups(a, first);
  const uint32_t jobs = (uint32_t)((int64_t)a.B * a.Hkv * a.num);  // a grid's threads are counted in 32 bits
  if (a.D == 256) return launch_cache_write_d<256>(a, c, grid, jobs, rest, st);
  if (a.D == 128) return launch_cache_write_d<128>(a, c, grid, jobs, rest, st);
  return launch_cache_write_d<64>(a, c, grid, jobs, rest, st);
}

}  // namespace kvx
