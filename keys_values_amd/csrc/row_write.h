// Rows of K and V to codes and to slots of a store, by the D / 8 adjacent lanes that hold a row: the quantiser and the slot write (quantize.hip), and the
// attention launch of a first chunk (sdpa_prefill.hip), which writes the chunk's rows beside its own work.
#pragma once
#include "kvx_common.h"

namespace kvx {
namespace {

constexpr int NTHREADS = 256;
constexpr int ROWS_PER_THREAD = 4;  // independent rows in flight per lane

// Reductions over the LPR (8, 16 or 32) adjacent lanes holding one row; every lane gets the result.
template <int LPR>
__device__ __forceinline__ float row_max(float v) {
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, true)));   // quad_perm [1,0,3,2]
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xf, 0xf, true)));   // quad_perm [2,3,0,1]
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xf, 0xf, true)));  // row_half_mirror
  if constexpr (LPR >= 16)
    v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xf, 0xf, true)));  // row_mirror
  if constexpr (LPR == 32) v = fmaxf(v, __shfl_xor(v, 16, 64));  // the other DPP row of the group
  return v;
}
template <int LPR>
__device__ __forceinline__ float row_min(float v) {
  v = fminf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, true)));
  v = fminf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xf, 0xf, true)));
  v = fminf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xf, 0xf, true)));
  if constexpr (LPR >= 16)
    v = fminf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xf, 0xf, true)));
  if constexpr (LPR == 32) v = fminf(v, __shfl_xor(v, 16, 64));
  return v;
}

// Does one of the 8 values hold a NaN? The reference takes a row's extremes with torch.aminmax
// (keys_values/kvcache/quantize/pytorch.py:90), which returns NaN for a row that holds one: such a row
// gets a NaN scale and dequantises to NaN throughout (fminf / fmaxf would drop the NaN).
__device__ __forceinline__ bool has_nan8(const float (&x)[8]) {
  return __builtin_isunordered(x[0], x[1]) | __builtin_isunordered(x[2], x[3]) | __builtin_isunordered(x[4], x[5]) |
         __builtin_isunordered(x[6], x[7]);
}

// True in all LPR lanes of a row if one of them says `bad`. The wavefront's ballot is a scalar: rows
// with a NaN are rare, and the test costs a scalar compare when there is none.
template <int LPR>
__device__ __forceinline__ bool row_any(bool bad) {
  const unsigned long long m = __ballot(bad);
  if (m == 0) return false;
  if constexpr (LPR == 64) return true;
  const int first = (int)(__lane_id() & ~(unsigned)(LPR - 1));
  return ((m >> first) & (~0ull >> (64 - LPR))) != 0;
}

// Codes of 4 values packed into a dword, byte e = clamp(rint(x[e] * inv) + zf, 0, 255). The sum is an
// integer-valued float, so the conversion's rounding does not matter; v_cvt_pk_u8_f32 saturates to
// [0, 255] (a NaN gives 0) and places the byte, which is the clamp, the cast and the packing in one.
__device__ __forceinline__ uint32_t codes4_u8(float x0, float x1, float x2, float x3, float inv, float zf) {
  uint32_t w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_rintf(x0 * inv) + zf, 0, 0);
  w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_rintf(x1 * inv) + zf, 1, w);
  w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_rintf(x2 * inv) + zf, 2, w);
  return __builtin_amdgcn_cvt_pk_u8_f32(__builtin_rintf(x3 * inv) + zf, 3, w);
}
// The same with codes clamped to [0, 15] (4-bit store).
__device__ __forceinline__ uint32_t codes4_u4(float x0, float x1, float x2, float x3, float inv, float zf) {
  uint32_t w = __builtin_amdgcn_cvt_pk_u8_f32(fminf(__builtin_rintf(x0 * inv) + zf, 15.0f), 0, 0);
  w = __builtin_amdgcn_cvt_pk_u8_f32(fminf(__builtin_rintf(x1 * inv) + zf, 15.0f), 1, w);
  w = __builtin_amdgcn_cvt_pk_u8_f32(fminf(__builtin_rintf(x2 * inv) + zf, 15.0f), 2, w);
  return __builtin_amdgcn_cvt_pk_u8_f32(fminf(__builtin_rintf(x3 * inv) + zf, 15.0f), 3, w);
}

template <int LPR, bool F16>
__device__ __forceinline__ void row_extremes(u32x4_t raw, float (&x)[8], float& mn, float& mx) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    x[2 * e] = elem_lo<F16>(raw[e]);
    x[2 * e + 1] = elem_hi<F16>(raw[e]);
  }
  mn = x[0];
  mx = x[0];
#pragma unroll
  for (int e = 1; e < 8; ++e) {
    mn = fminf(mn, x[e]);
    mx = fmaxf(mx, x[e]);
  }
  mn = row_min<LPR>(mn);
  mx = row_max<LPR>(mx);
  if (row_any<LPR>(has_nan8(x))) mn = mx = __builtin_nanf("");
}

// The ROWS_PER_THREAD rows a lane works on at once share the per-row arithmetic (three IEEE divisions):
// all lanes of a row hold its extremes, so lane c of a quad works out the scale and zero point of row
// c only, and the others fetch 1 / scale and the zero point from it with a quad broadcast. Returns the
// codes of row i in c[i] (bytes), and in (scale, zp) the state of row (lane & 3).
template <int LPR, int BITS, bool F16>
__device__ __forceinline__ void quantize_rows_in_flight(const u32x4_t (&raw)[ROWS_PER_THREAD], u32x2_t (&c)[ROWS_PER_THREAD], float& scale,
                                                        int32_t& zp) {
  static_assert(ROWS_PER_THREAD == 4, "one row per lane of a quad");
  float x[ROWS_PER_THREAD][8], mn[ROWS_PER_THREAD], mx[ROWS_PER_THREAD];
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD; ++i) row_extremes<LPR, F16>(raw[i], x[i], mn[i], mx[i]);
  const int mine = (int)(__lane_id() & 3u);
  const float my_mn = mine == 0 ? mn[0] : mine == 1 ? mn[1] : mine == 2 ? mn[2] : mn[3];
  const float my_mx = mine == 0 ? mx[0] : mine == 1 ? mx[1] : mine == 2 ? mx[2] : mx[3];
  quant_params(my_mn, my_mx, scale, zp, BITS == 8 ? 255.0f : 15.0f);
  const int inv_bits = __builtin_bit_cast(int, 1.0f / scale);
  const int zf_bits = __builtin_bit_cast(int, (float)zp);
  float inv[ROWS_PER_THREAD], zf[ROWS_PER_THREAD];
  inv[0] = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(inv_bits, 0x00, 0xf, 0xf, true));  // quad_perm [0,0,0,0]
  inv[1] = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(inv_bits, 0x55, 0xf, 0xf, true));  // quad_perm [1,1,1,1]
  inv[2] = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(inv_bits, 0xAA, 0xf, 0xf, true));  // quad_perm [2,2,2,2]
  inv[3] = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(inv_bits, 0xFF, 0xf, 0xf, true));  // quad_perm [3,3,3,3]
  zf[0] = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(zf_bits, 0x00, 0xf, 0xf, true));
  zf[1] = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(zf_bits, 0x55, 0xf, 0xf, true));
  zf[2] = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(zf_bits, 0xAA, 0xf, 0xf, true));
  zf[3] = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(zf_bits, 0xFF, 0xf, 0xf, true));
#pragma unroll
  for (int i = 0; i < ROWS_PER_THREAD; ++i) {
    if constexpr (BITS == 8) {
      c[i][0] = codes4_u8(x[i][0], x[i][1], x[i][2], x[i][3], inv[i], zf[i]);
      c[i][1] = codes4_u8(x[i][4], x[i][5], x[i][6], x[i][7], inv[i], zf[i]);
    } else {
      c[i][0] = codes4_u4(x[i][0], x[i][1], x[i][2], x[i][3], inv[i], zf[i]);
      c[i][1] = codes4_u4(x[i][4], x[i][5], x[i][6], x[i][7], inv[i], zf[i]);
    }
  }
}

// Quantise the 8 values of this lane's share of a K and a V row. Even lanes work out the scale and zero point of the K row, odd ones of
// the V row, and each fetches 1 / scale and the zero point of the other from its neighbour; (scale, zp): the lane's own row's.
template <int LPR, bool F16>
__device__ __forceinline__ void quantize8_kv(const u32x4_t& k, const u32x4_t& v, u32x2_t& kc, u32x2_t& vc, float& scale, int32_t& zp) {
  float xk[8], xv[8], mnk, mxk, mnv, mxv;
  row_extremes<LPR, F16>(k, xk, mnk, mxk);
  row_extremes<LPR, F16>(v, xv, mnv, mxv);
  const bool odd = __lane_id() & 1u;
  quant_params(odd ? mnv : mnk, odd ? mxv : mxk, scale, zp);
  const int inv = __builtin_bit_cast(int, 1.0f / scale), zf = __builtin_bit_cast(int, (float)zp);
  auto of_k = [](int x) { return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(x, 0xA0, 0xf, 0xf, true)); };  // quad_perm [0,0,2,2]
  auto of_v = [](int x) { return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(x, 0xF5, 0xf, 0xf, true)); };  // quad_perm [1,1,3,3]
  const float ik = of_k(inv), zk = of_k(zf), iv = of_v(inv), zv = of_v(zf);
  kc = u32x2_t{codes4_u8(xk[0], xk[1], xk[2], xk[3], ik, zk), codes4_u8(xk[4], xk[5], xk[6], xk[7], ik, zk)};
  vc = u32x2_t{codes4_u8(xv[0], xv[1], xv[2], xv[3], iv, zv), codes4_u8(xv[4], xv[5], xv[6], xv[7], iv, zv)};
}

// Codes of the lane's 8 values as bytes (0..15), in the layout of quantize8_kv.
template <int LPR, bool F16>
__device__ __forceinline__ u32x2_t quantize4(u32x4_t raw, float& scale, int32_t& zp) {
  float x[8];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    x[2 * e] = elem_lo<F16>(raw[e]);
    x[2 * e + 1] = elem_hi<F16>(raw[e]);
  }
  float mn = x[0], mx = x[0];
#pragma unroll
  for (int e = 1; e < 8; ++e) {
    mn = fminf(mn, x[e]);
    mx = fmaxf(mx, x[e]);
  }
  mn = row_min<LPR>(mn);
  mx = row_max<LPR>(mx);
  if (row_any<LPR>(has_nan8(x))) mn = mx = __builtin_nanf("");  // aminmax propagates NaN, fminf / fmaxf drop it
  quant_params(mn, mx, scale, zp, 15.0f);
  const float inv = 1.0f / scale;
  const float zf = (float)zp;
  u32x2_t out;
  out[0] = quant_code(x[0], inv, zf, 15.0f) | (quant_code(x[1], inv, zf, 15.0f) << 8) | (quant_code(x[2], inv, zf, 15.0f) << 16) |
           (quant_code(x[3], inv, zf, 15.0f) << 24);
  out[1] = quant_code(x[4], inv, zf, 15.0f) | (quant_code(x[5], inv, zf, 15.0f) << 8) | (quant_code(x[6], inv, zf, 15.0f) << 16) |
           (quant_code(x[7], inv, zf, 15.0f) << 24);
  return out;
}

// Sum over the LPR adjacent lanes holding one row; every lane gets the result.
template <int LPR>
__device__ __forceinline__ float row_sum(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, true));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xf, 0xf, true));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xf, 0xf, true));
  if constexpr (LPR >= 16)
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xf, 0xf, true));
  if constexpr (LPR == 32) v += __shfl_xor(v, 16, 64);  // the other DPP row of the group
  return v;
}

// |row|_2 of a bf16 (F16: fp16) row spread over LPR lanes, accumulated in fp32.
template <int LPR, bool F16 = false>
__device__ __forceinline__ float row_norm(u32x4_t raw) {
  float ss = 0.0f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float a = elem_lo<F16>(raw[e]), b = elem_hi<F16>(raw[e]);
    ss += a * a;
    ss += b * b;
  }
  return sqrtf(row_sum<LPR>(ss));
}

// |x - dq(q(x))|_2 of a row: the dequantised value and the difference are rounded to the rows' type, the norm
// accumulates in fp32 (keys_values/kvcache/quantize/pytorch.py:530-548).
template <int LPR, bool F16>
__device__ __forceinline__ float row_quant_error(u32x4_t raw, u32x2_t codes, float scale, int32_t zp) {
  float ss = 0.0f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t cw = codes[e >> 1];
    const int sh = (e & 1) * 16;
    const uint32_t dq = dequant_pair<F16>((cw >> sh) & 0xff, (cw >> (sh + 8)) & 0xff, zp, scale);
    const uint32_t diff = pack_pair<F16>(elem_lo<F16>(raw[e]) - elem_lo<F16>(dq), elem_hi<F16>(raw[e]) - elem_hi<F16>(dq));
    const float a = elem_lo<F16>(diff), b = elem_hi<F16>(diff);
    ss += a * a;
    ss += b * b;
  }
  return sqrtf(row_sum<LPR>(ss));
}

// A quantised store: quantise the rows held as (krow, vrow) by the lanes of a job and store them in slot `target`; kc_row, vc_row: the lane's place in slot
// 0. Every lane of the wavefront calls it (the row reductions need all lanes of a row). Returns the rows' quantisation errors.
template <int D, int KV>
__device__ __forceinline__ float put_rows(const kvx_cache_write_args& a, uint8_t* kc_row, uint8_t* vc_row, int64_t qs_row, int col, const u32x4_t& krow, const u32x4_t& vrow,
                                          int target, bool doit, bool want_err) {
  constexpr bool U4 = kv_is_u4(KV), F16 = kv_elem_f16(KV);
  constexpr int LPR = D / 8;
  float s1, s2, err = 0.0f;
  int32_t z1, z2;
  u32x2_t kc, vc;
  if constexpr (U4) {
    kc = quantize4<LPR, F16>(krow, s1, z1);
    vc = quantize4<LPR, F16>(vrow, s2, z2);
  } else {
    float s;
    int32_t z;
    quantize8_kv<LPR, F16>(krow, vrow, kc, vc, s, z);
    s1 = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, s), 0xA0, 0xf, 0xf, true));
    s2 = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, s), 0xF5, 0xf, 0xf, true));
    z1 = __builtin_amdgcn_mov_dpp(z, 0xA0, 0xf, 0xf, true);
    z2 = __builtin_amdgcn_mov_dpp(z, 0xF5, 0xf, 0xf, true);
  }
  if (want_err) err = row_quant_error<LPR, F16>(krow, kc, s1, z1) + row_quant_error<LPR, F16>(vrow, vc, s2, z2);  // uniform branch
  if constexpr (U4) {  // byte j = code[j] << 4 | code[j + D/2]: the partner lane holds the low nibbles
    kc = u32x2_t{(kc[0] << 4) | (uint32_t)__shfl_xor(kc[0], LPR / 2, 64), (kc[1] << 4) | (uint32_t)__shfl_xor(kc[1], LPR / 2, 64)};
    vc = u32x2_t{(vc[0] << 4) | (uint32_t)__shfl_xor(vc[0], LPR / 2, 64), (vc[1] << 4) | (uint32_t)__shfl_xor(vc[1], LPR / 2, 64)};
  }
  if (doit) {
    if (!U4 || col < LPR / 2) {
      *(u32x2_t*)(kc_row + (int64_t)target * a.kc_stride_t) = kc;
      *(u32x2_t*)(vc_row + (int64_t)target * a.vc_stride_t) = vc;
    }
    if (col == 0) {
      a.k_scale[qs_row + target] = s1;
      a.k_zp[qs_row + target] = z1;
      a.v_scale[qs_row + target] = s2;
      a.v_zp[qs_row + target] = z2;
    }
  }
  return err;
}

// Tokens [t0, t1) of pair (b, hh) of a first chunk, by a workgroup of NTHREADS: what cache_write_kernel does with them (no ring, no log). Four of a lane's
// jobs are in flight.
template <int D, int KV>
__device__ __forceinline__ void write_tokens(const kvx_cache_write_args& a, int b, int hh, int t0, int t1) {
  constexpr bool PLAIN = kv_is_plain(KV), U4 = kv_is_u4(KV), F16 = kv_elem_f16(KV);
  constexpr int LPR = D / 8, JOBS = NTHREADS / LPR, N = 4, ES = PLAIN ? 2 : 1;
  const int col = threadIdx.x % LPR, ccol = U4 ? col % (LPR / 2) : col;
  const int64_t sc_row = b * a.sc_stride_b + hh * a.sc_stride_h;
  uint8_t* kc_row = (uint8_t*)a.k_cache + (b * a.kc_stride_b + hh * a.kc_stride_h) * ES + ccol * 8 * ES;
  uint8_t* vc_row = (uint8_t*)a.v_cache + (b * a.vc_stride_b + hh * a.vc_stride_h) * ES + ccol * 8 * ES;
  for (int first = t0 + (int)threadIdx.x / LPR; first - (int)threadIdx.x / LPR < t1; first += N * JOBS) {  // all lanes stay: rows are reduced across them
    u32x4_t kr[N], vr[N];
    int slot[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int j = min(first + i * JOBS, t1 - 1);
      kr[i] = *(const u32x4_t*)((const uint16_t*)a.key + b * a.key_stride_b + hh * a.key_stride_h + (int64_t)j * a.key_stride_t + col * 8);
      vr[i] = *(const u32x4_t*)((const uint16_t*)a.value + b * a.value_stride_b + hh * a.value_stride_h + (int64_t)j * a.value_stride_t + col * 8);
      slot[i] = a.index[b * a.index_stride_b + hh * a.index_stride_h + j];
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      if (first - (int)threadIdx.x / LPR + i * JOBS >= t1) break;  // nobody has a job: uniform
      const int j = first + i * JOBS;
      const bool ok = j < t1 && slot[i] >= 0 && slot[i] < a.cache_len;  // a bad index is dropped, never written out of bounds
      float err = 0.0f, norm = 0.0f;
      if constexpr (PLAIN) {
        if (ok) {
          *(u32x4_t*)(kc_row + (int64_t)slot[i] * a.kc_stride_t * ES) = kr[i];
          *(u32x4_t*)(vc_row + (int64_t)slot[i] * a.vc_stride_t * ES) = vr[i];
        }
      } else {
        err = put_rows<D, KV>(a, kc_row, vc_row, b * a.qs_stride_b + hh * a.qs_stride_h, col, kr[i], vr[i], slot[i], ok, a.q_errors != nullptr);
      }
      if (a.v_norm) norm = row_norm<LPR, F16>(vr[i]);
      if (ok && col == 0) {
        if (a.token_pos) a.token_pos[b * a.tp_stride_b + hh * a.tp_stride_h + slot[i]] = a.input_pos + j;
        if (a.scores) a.scores[sc_row + slot[i]] = 0.0f;
        if (a.v_norm) a.v_norm[sc_row + slot[i]] = norm;
        if (a.q_errors) a.q_errors[sc_row + slot[i]] = err;
      }
    }
  }
}

}  // namespace
}  // namespace kvx
