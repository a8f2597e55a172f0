// Arguments of the attention kernels for chunks: the tiled one (sdpa_prefill.hip) and the one for few rows (sdpa_rows.hip).
#pragma once
#include "prefill_merge.h"

namespace kvx {

constexpr int BN = 64;  // keys per tile; splits are whole tiles

struct PrefillParams {
  const uint16_t* q;
  const void* k;
  const void* v;
  const float* k_scale;
  const int32_t* k_zp;
  const float* v_scale;
  const int32_t* v_zp;
  const int32_t* tp;
  uint16_t* o;
  float* lse;
  float* part_o;   // [split][group][R][D] fp32, unnormalised
  float* part_ml;  // [split][team][group][R][2]  (max in log2 units, sum)
  int32_t B, Hq, Hkv, G, q_len, kv_len, R, input_pos;
  int32_t num_splits, tiles_per_split, num_tiles, m_blocks;
  int32_t period;  // a causal first chunk in splits: blocks of rows that a split's keys cover, 0: all splits of all rows
  int32_t pair;    // two teams of a workgroup walk the halves of a split
  float c;  // sm_scale * log2(e)
  int64_t q_sb, q_sh, q_st, k_sb, k_sh, k_st, v_sb, v_sh, v_st, o_sb, o_sh, o_st;
  int64_t qs_sb, qs_sh, tp_sb, tp_sh;
  int32_t columns;  // rows a workgroup of the kernel for few rows (sdpa_rows.hip), 0: the tiled kernel
  int32_t qs_vec, tp_vec;  // quantiser state / positions may be read four keys at a time
};

// How the kernel for few rows takes a call: rows of a workgroup (16 or 32; 0: the call keeps the tiled kernel), KV splits, estimated ns
struct RowsPlan {
  int columns, splits;
  int64_t ns;
};
// `combined`: the score-sum launch that follows combines the splits
RowsPlan rows_plan(const kvx_sdpa_args& a, bool combined);
int launch_sdpa_rows(const PrefillParams& p, int D, int kv, hipStream_t st);
void common_params(PrefillParams& p, const kvx_sdpa_args& a);
int64_t prefill_ns(const kvx_sdpa_args& a);  // estimate of a call's attention launch where a score-sum launch follows

}  // namespace kvx
