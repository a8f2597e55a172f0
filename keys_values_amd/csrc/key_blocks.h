// Blocks of 32 keys as operands of v_mfma_f32_16x16x32, straight from memory: K rows as the A operands of S^T = K Q^T (16 keys a
// tile), V rows as those of O^T = V^T P^T (32 keys). Shared by the kernels that keep their query rows in registers and stream the keys
// past them: single tokens (sdpa_decode.h) and chunks of few rows (sdpa_rows.hip).
//
// The lane that holds key m of a tile loads 8 consecutive d of that row per matrix instruction: the row as it lies in memory, or its
// dequantised codes, is the A operand. The accumulator layout of S^T (lane = column, keys 4 kg .. 4 kg + 3 of lane group kg)
// becomes the B operand of the second product once the 32 keys of a block are taken in the order (tile 0: 4 kg .. 4 kg + 3, tile 1:
// 4 kg .. 4 kg + 3) per lane group; V^T is gathered to match: a lane loads, from each of its 8 keys, the D / 16 values of its d rows
// and regroups them (one byte permute per pair of plain values; for codes the regrouping is part of the dequantisation).
#pragma once
#include "kvx_common.h"

namespace kvx {

template <bool F16>
__device__ __forceinline__ f32x4_t mfma_16x16x32(u32x4_t a, u32x4_t b, f32x4_t c) {
  if constexpr (F16) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// elem( (float)((int)code - zp) * scale ) for two codes with their own row state (two keys)
template <bool F16>
__device__ __forceinline__ uint32_t dequant_pair2(uint32_t c0, int32_t zp0, float sc0, uint32_t c1, int32_t zp1, float sc1) {
  return pack_pair<F16>((float)((int32_t)c0 - zp0) * sc0, (float)((int32_t)c1 - zp1) * sc1);
}

// NT: rows are read once by the launch, past the caches. Rows are addressed from a uniform base by 32-bit byte offsets (the host
// checks the range).
template <int D, int KV, bool NT>
struct KeyBlocks {
  static constexpr bool F16 = kv_elem_f16(KV);
  static constexpr bool U8 = !kv_is_plain(KV);  // codes + row state (8-bit or 4-bit store)
  static constexpr bool U4 = kv_is_u4(KV);
  static constexpr int KJ = D / 32;   // matrix instructions of the first product per 16-key tile
  static constexpr int DPL = D / 16;  // d rows per lane = matrix instructions of the second product per 32-key block
  static constexpr int CH = 32;       // keys of a block
  static constexpr int NL4 = D >= 128 ? D / 128 : 1;                              // 4-bit rows: 16-byte loads per key of K
  static constexpr int KR = U4 ? NL4 : (U8 ? D / 64 : KJ);                        // 16-byte loads per key of K
  static constexpr int VW = U4 ? (DPL + 7) / 8 : (U8 ? (DPL + 3) / 4 : DPL / 2);  // dwords per key of V
  static_assert(D == 64 || D == 128 || (D == 256 && U8), "plain rows of 256 values do not fit the registers");

  // first d of the 8 that lane group kg supplies to matrix instruction e of the first product
  __device__ __forceinline__ static int kslice(int e, int kg) {
    if constexpr (!U8) return 8 * (kg + 4 * e);
    else if constexpr (U4 && D == 64) return 8 * kg + 32 * e;
    else if constexpr (U4) return 16 * kg + 8 * (e & 1) + 64 * ((e >> 1) % NL4) + (D / 2) * (e / (2 * NL4));
    else return 16 * kg + 8 * (e & 1) + 64 * (e >> 1);
  }
  // d of row `mrow` of matrix instruction t of the second product
  __device__ __forceinline__ static int dmap(int t, int mrow) {
    if constexpr (U4) return t < DPL / 2 ? (DPL / 2) * mrow + t : D / 2 + (DPL / 2) * mrow + (t - DPL / 2);
    else return DPL * mrow + t;
  }

  struct Rows {
    u32x4_t k[2][KR];
    float ks[2];
    int32_t kz[2];
    uint32_t v[8][VW];
    float vs[8];
    int32_t vz[8];
  };

  const uint8_t *kbase, *vbase;
  uint32_t k_rowb, v_rowb, k_lane, v_lane, k16, v16;
  const char *ksb, *kzb, *vsb, *vzb;
  bool qs_vec;  // quantiser state arrays are 16-byte aligned with strides that keep them so
  int m, kg, k_end;

  // k_off, v_off, qs_off, k_st, v_st: elements
  __device__ __forceinline__ void init(const void* k, const void* v, const float* k_scale, const int32_t* k_zp, const float* v_scale, const int32_t* v_zp, int64_t k_off,
                                       int64_t v_off, int64_t qs_off, int64_t k_st, int64_t v_st, bool vec, int m_, int kg_, int k_end_) {
    constexpr int ES = U8 ? 1 : 2;
    m = m_;
    kg = kg_;
    k_end = k_end_;
    kbase = (const uint8_t*)k + k_off * ES;
    vbase = (const uint8_t*)v + v_off * ES;
    k_rowb = (uint32_t)k_st * ES;
    v_rowb = (uint32_t)v_st * ES;
    k_lane = (U4 && D == 64) ? 8 * kg : 16 * kg;  // + 64 r for the r-th load of the row
    v_lane = (uint32_t)m * (U4 ? DPL / 2 : (U8 ? DPL : 2 * DPL));
    k16 = 16u * k_rowb;
    v16 = 16u * v_rowb;
    ksb = (const char*)(k_scale + qs_off);
    kzb = (const char*)(k_zp + qs_off);
    vsb = (const char*)(v_scale + qs_off);
    vzb = (const char*)(v_zp + qs_off);
    qs_vec = vec;
  }

  // The calls ask for slot, head and batch strides of whole 8 elements: rows of codes begin on 8 bytes, plain ones on 16. A wider load
  // of codes says so (the same instruction: global loads of 16 bytes need no more than 4).
  template <typename T>
  __device__ __forceinline__ static T get(const void* p) {
    constexpr size_t ALIGN = U8 && sizeof(T) > 8 ? 8 : sizeof(T);
    typedef T row_part __attribute__((aligned(ALIGN)));
    if constexpr (NT) return __builtin_nontemporal_load((const row_part*)p);
    else return *(const row_part*)p;
  }
  __device__ __forceinline__ void load_k(Rows& r, int gi, uint32_t off, int key) const {
    const uint8_t* row = kbase + off;
#pragma unroll
    for (int x = 0; x < KR; ++x) {
      if constexpr (U4 && D == 64) {
        const u32x2_t c = get<u32x2_t>(row);
        r.k[gi][x] = u32x4_t{c[0], c[1], 0u, 0u};
      } else {
        r.k[gi][x] = get<u32x4_t>(row + 64 * x);
      }
    }
    if constexpr (U8) {  // uniform base + 32-bit offset
      r.ks[gi] = *(const float*)(ksb + (uint32_t)key * 4u);
      r.kz[gi] = *(const int32_t*)(kzb + (uint32_t)key * 4u);
    }
  }
  __device__ __forceinline__ void load_v(Rows& r, int j, uint32_t off) const {
    const uint8_t* row = vbase + off;
    constexpr int BYTES = U4 ? DPL / 2 : (U8 ? DPL : 2 * DPL);  // this lane's share of the row
    if constexpr (BYTES == 16) {
      const u32x4_t x = get<u32x4_t>(row);
      r.v[j][0] = x[0]; r.v[j][1] = x[1]; r.v[j][2] = x[2]; r.v[j][3] = x[3];
    } else if constexpr (BYTES == 8) {
      const u32x2_t x = get<u32x2_t>(row);
      r.v[j][0] = x[0]; r.v[j][1] = x[1];
    } else if constexpr (BYTES == 4) {
      r.v[j][0] = get<uint32_t>(row);
    } else {
      static_assert(BYTES == 2, "4-bit rows of 64 values");
      r.v[j][0] = (uint32_t)get<uint16_t>(row);
    }
  }
  // This lane's rows of the block at `chunk0`: K rows chunk0 + m and chunk0 + 16 + m, V rows chunk0 + 4 kg (+ 0..3, + 16..19). A
  // full block addresses them from two per-lane offsets that advance with the block and multiples of the row stride; a block that
  // reaches past the end clamps every key to the last valid row (its logits are to become -inf).
  __device__ __forceinline__ void issue(Rows& r, int chunk0) const {
    if (chunk0 + CH <= k_end) {
      const uint32_t ko = (uint32_t)(chunk0 + m) * k_rowb + k_lane;
      load_k(r, 0, ko, chunk0 + m);
      load_k(r, 1, ko + k16, chunk0 + 16 + m);
      const int q0 = chunk0 + 4 * kg;
      if constexpr (U8) {
        if (qs_vec) {  // the four keys of a tile this lane group owns are neighbours: one 16-byte load each
#pragma unroll
          for (int gi = 0; gi < 2; ++gi) {
            const f32x4_t sc = *(const f32x4_t*)(vsb + (uint32_t)(q0 + 16 * gi) * 4u);
            const int4 zp = *(const int4*)(vzb + (uint32_t)(q0 + 16 * gi) * 4u);
            r.vs[4 * gi] = sc[0]; r.vs[4 * gi + 1] = sc[1]; r.vs[4 * gi + 2] = sc[2]; r.vs[4 * gi + 3] = sc[3];
            r.vz[4 * gi] = zp.x; r.vz[4 * gi + 1] = zp.y; r.vz[4 * gi + 2] = zp.z; r.vz[4 * gi + 3] = zp.w;
          }
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            r.vs[j] = *(const float*)(vsb + (uint32_t)(q0 + 16 * (j >> 2) + (j & 3)) * 4u);
            r.vz[j] = *(const int32_t*)(vzb + (uint32_t)(q0 + 16 * (j >> 2) + (j & 3)) * 4u);
          }
        }
      }
      const uint32_t vo = (uint32_t)q0 * v_rowb + v_lane;
#pragma unroll
      for (int j = 0; j < 8; ++j) load_v(r, j, vo + (uint32_t)(j & 3) * v_rowb + (j >> 2) * v16);
    } else {
#pragma unroll
      for (int gi = 0; gi < 2; ++gi) {
        const int key = min(chunk0 + 16 * gi + m, k_end - 1);
        load_k(r, gi, (uint32_t)key * k_rowb + k_lane, key);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = min(chunk0 + 16 * (j >> 2) + 4 * kg + (j & 3), k_end - 1);
        if constexpr (U8) {
          r.vs[j] = *(const float*)(vsb + (uint32_t)key * 4u);
          r.vz[j] = *(const int32_t*)(vzb + (uint32_t)key * 4u);
        }
        load_v(r, j, (uint32_t)key * v_rowb + v_lane);
      }
    }
  }
  // A operand e of the first product for tile gi
  __device__ __forceinline__ static u32x4_t k_operand(const Rows& r, int gi, int e) {
    if constexpr (!U8) {
      return r.k[gi][e];
    } else if constexpr (!U4) {
      const u32x4_t w = r.k[gi][e >> 1];
      return (e & 1) ? dequant_words<F16>(w[2], w[3], r.kz[gi], r.ks[gi]) : dequant_words<F16>(w[0], w[1], r.kz[gi], r.ks[gi]);
    } else {
      const u32x4_t w = r.k[gi][D >= 128 ? (e >> 1) % NL4 : 0];
      u32x2_t bytes;
      int shift;
      if constexpr (D >= 128) {
        bytes = (e & 1) ? u32x2_t{w[2], w[3]} : u32x2_t{w[0], w[1]};
        shift = (e / (2 * NL4)) ? 0 : 4;
      } else {
        bytes = u32x2_t{w[0], w[1]};
        shift = e ? 0 : 4;
      }
      const u32x2_t c = u4_codes(bytes, shift);
      return dequant_words<F16>(c[0], c[1], r.kz[gi], r.ks[gi]);
    }
  }
  // A operand t of the second product: value t of each of this lane's 8 keys, in key order
  __device__ __forceinline__ static u32x4_t v_operand(const Rows& r, int t) {
    u32x4_t a;
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const int j0 = 2 * jj, j1 = 2 * jj + 1;
      if constexpr (!U8) {
        a[jj] = __builtin_amdgcn_perm(r.v[j1][t >> 1], r.v[j0][t >> 1], (t & 1) ? 0x07060302u : 0x05040100u);
      } else {
        uint32_t c0, c1;
        if constexpr (!U4) {
          c0 = (r.v[j0][t >> 2] >> (8 * (t & 3))) & 0xffu;
          c1 = (r.v[j1][t >> 2] >> (8 * (t & 3))) & 0xffu;
        } else {
          const int tb = t < DPL / 2 ? t : t - DPL / 2;  // byte of this lane's share; first half of the row: high nibble
          const int sh = 8 * (tb & 3) + (t < DPL / 2 ? 4 : 0);
          c0 = (r.v[j0][tb >> 2] >> sh) & 0xfu;
          c1 = (r.v[j1][tb >> 2] >> sh) & 0xfu;
        }
        a[jj] = dequant_pair2<F16>(c0, r.vz[j0], r.vs[j0], c1, r.vz[j1], r.vs[j1]);
      }
    }
    return a;
  }
};

}  // namespace kvx
