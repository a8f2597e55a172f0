// Single-token decode attention: how a call is cut into splits, where its workspace keeps what, and the launches of a step.
// The kernels are in sdpa_decode.h.
#include "sdpa_decode.h"

#include <stdlib.h>

#include <atomic>
#include <mutex>

namespace kvx {
namespace {

using namespace decode;

// Before the split kernel, where the slot write does not do it: no split of a row has published or arrived, no row has a
// lowest-score slot yet.
__global__ void decode_init_kernel(const DecodeCounters c, unsigned long long* best, uint32_t* tail_count, int rows, uint32_t scratch_splits_init) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  clear_counters(c, i, gridDim.x * blockDim.x, rows);
  if (i < rows && best) best[i] = ~0ull;
  if (i == 0 && tail_count) *tail_count = 0u;
  if (i == 0 && c.scratch_splits) *c.scratch_splits = scratch_splits_init;
}

struct Plan {
  int G, num_splits, keys_per_split, Tpad, resident, one_launch;
  size_t off_logits, off_part_o, off_part_ml, off_part_best, off_part_vn, off_part_stats, off_pending, off_best, off_tail, off_count, total;
};

// Switches of the route the logits take, process-wide. Defaults come from the environment, read ONCE (first use):
// KVX_DECODE_RESIDENT=0 sends every split's logits through the scratch; KVX_DECODE_SPIN_LIMIT bounds the wait for a
// row's other splits in polls (0: no wait, every workgroup takes the scratch route); KVX_DECODE_POLL_SLEEP is the
// pause between two polls in units of 512 cycles. kvx_decode_tuning() replaces them at run time. Values are clamped:
// the longest wait a workgroup can spend is spin_limit x (poll_sleep x 512 + a load's latency) cycles, i.e.
// 2^20 x 64 x 512 cycles = 16 s at the clamps and about 30 ms at the defaults (2^15 polls, 4 x 512 cycles).
constexpr int kSpinDefault = 1 << 15, kSpinMax = 1 << 20, kSleepDefault = 4, kSleepMax = 64;
struct Tuning {
  std::atomic<int> resident{1}, spin_limit{kSpinDefault}, poll_sleep{kSleepDefault};
  int env_resident = 1, env_spin = kSpinDefault, env_sleep = kSleepDefault;
};
int clampi(int x, int lo, int hi) { return x < lo ? lo : (x > hi ? hi : x); }
int env_int(const char* name, int dflt) {
  const char* e = getenv(name);
  if (!e || !*e) return dflt;
  char* end = nullptr;
  const long v = strtol(e, &end, 10);
  return (end == e || *end) ? dflt : (int)(v < -1 ? -1 : (v > (1l << 30) ? (1l << 30) : v));  // not a number: the default
}
Tuning& tuning() {
  static Tuning t;
  static std::once_flag once;
  std::call_once(once, [] {
    t.env_resident = env_int("KVX_DECODE_RESIDENT", 1) != 0;
    t.env_spin = clampi(env_int("KVX_DECODE_SPIN_LIMIT", kSpinDefault), 0, kSpinMax);
    t.env_sleep = clampi(env_int("KVX_DECODE_POLL_SLEEP", kSleepDefault), 0, kSleepMax);
    t.resident = t.env_resident;
    t.spin_limit = t.env_spin;
    t.poll_sleep = t.env_sleep;
  });
  return t;
}

Plan make_plan(const kvx_sdpa_args& a, bool fused_h2o) {
  Plan pl;
  const int gr = a.Hq / a.Hkv;
  pl.G = gr <= 1 ? 1 : (gr <= 2 ? 2 : (gr <= 4 ? 4 : (gr <= 8 ? 8 : 16)));
  // Splits: as many as give every compute unit one workgroup and not one more (a few workgroups too many are a second
  // round for everybody: 16 rows of 35407 8-bit keys at head size 256 in 17 splits took 137 us, in 16 they take 80), of at
  // least 128 keys (a wavefront's steps take about 1 us each; shorter splits only add partials to combine), at most 128
  // a row (64 below 16384 keys: the splits of a row wait for each other), and with weights no longer than what the LDS
  // holds of a split's logits (long rows of many heads then run several full rounds). Two workgroups per compute unit, as
  // many as fit, were worse wherever one round covers the call. Measured, us, two -> one per compute unit: 8 rows of
  // 16384 keys 25.0 -> 21.4, of 65536 keys 55 -> 50, 32 rows of 16384 keys 52.6 -> 49.8; 8-bit codes 8 rows of 32768 keys
  // 29 -> 25; head size 256, 8-bit codes, 32 rows of 8192 keys 49 -> 40; 8 rows of 1024 keys, 256 -> 128 keys a split
  // 13.1 -> 11.8. 64 rows of 32768 keys take 170 in two rounds of 4096 keys, 183 in splits of 1024.
  const bool weights = a.w || fused_h2o;
  const int allow_resident = weights ? tuning().resident.load() : 0;
  const int lgk = logit_floats(pl.G, a.D, !kv_is_plain(a.kv_dtype)) / pl.G;
  int splits = a.num_splits;
  if (splits <= 0) {
    const int64_t rows = (int64_t)a.B * a.Hkv, cus = num_cus();
    auto in_rounds = [&](int64_t r) { return max((int64_t)1, r * cus / rows); };  // splits of r rounds of one workgroup per compute unit
    int64_t n = in_rounds(1);
    // codes are bound by the vector arithmetic of their dequantisation: long splits gain from a second workgroup a unit
    // (32 rows of 16384 keys, 4 bits: 33 us against 36)
    if (!kv_is_plain(a.kv_dtype) && a.D <= 128 && a.kv_len / n > 1024) n = min(in_rounds(2), max(n, (int64_t)a.kv_len / 1024));
    n = min(n, min((int64_t)(a.kv_len + 127) / 128, (int64_t)(a.kv_len < 16384 ? 64 : 128)));
    if (allow_resident && a.kv_len > n * lgk) {
      const int64_t least = (a.kv_len + lgk - 1) / lgk;
      // More than 256 splits a row (head size 64: 8 heads from 524289 keys on, 16 from 196609) only where the device holds all of
      // the call's at once. Through the scratch -> on the chip, us: one row of 16 heads over 197000 keys 37 -> 34, 393216
      // 50 -> 42, of 8 heads over 600000 61 -> 47; two rows of 16 heads over 197000 keys 41 -> 61, over 393216 68 -> 81, four
      // rows over 262144 8-bit keys 66 -> 115.
      // Rows whose logits fit the chip in no 512 splits go through the scratch anyway: one workgroup per compute unit, also for a
      // single row, whose 128 splits would use half the device. 128 -> 256 splits, us: one row of 16 heads of 64 over 600000 keys
      // 70 -> 66, over 1.5 M 155 -> 126, of 128 over 300000 62 -> 59, over 600000 108 -> 93, 8 of 128 over 950000 151 -> 118; 512
      // splits: 83, 139, 76, 112, 136.
      const bool fits = least <= kMaxSplits && (least <= WAVES * a.D || least * rows <= 2 * cus);
      n = fits ? max(least, in_rounds((least * rows + cus - 1) / cus)) : max(n, in_rounds(1));
    }
    splits = (int)min(n, (int64_t)kMaxSplits);
  }
  splits = max(1, min(splits, kMaxSplits));
  int kps = (a.kv_len + splits - 1) / splits;
  kps = ((kps + 63) / 64) * 64;  // keeps the chunks of a split aligned to the logits rows
  pl.keys_per_split = kps;
  pl.num_splits = (a.kv_len + kps - 1) / kps;
  pl.Tpad = ((a.kv_len + 63) / 64) * 64;
  // The splits of a row wait for each other: they have to fit the device side by side (workgroups are dispatched in index
  // order, a row's splits are neighbours). At head size 256 a compute unit holds one workgroup, else two.
  const bool side_by_side = pl.num_splits <= (a.D > 128 ? 1 : 2) * num_cus();
  pl.resident = allow_resident && kps <= lgk && side_by_side;
  pl.one_launch = side_by_side && (pl.resident || !weights);
  size_t off = 0;
  auto take = [&off](size_t bytes) {  // 16-byte aligned pieces
    const size_t at = off;
    off += (bytes + 15) & ~(size_t)15;
    return at;
  };
  const size_t rows = (size_t)a.B * a.Hkv, row_splits = rows * pl.num_splits, head_splits = (size_t)a.B * a.Hq * pl.num_splits;
  const bool fused_one = fused_h2o && pl.one_launch, fused_two = fused_h2o && !pl.one_launch;
  pl.off_logits = take(weights ? rows * pl.G * pl.Tpad * 4 : 0);
  pl.off_part_o = take(head_splits * a.D * 4);
  pl.off_part_ml = take(head_splits * 2 * 4);
  // the choice after the combination with the errors hands its minima over in the same place
  pl.off_part_best = take(fused_one ? rows * max(pl.num_splits, select_one_parts(a.kv_len)) * 8 : 0);
  pl.off_part_vn = take(fused_one ? head_splits * 4 : 0);
  pl.off_part_stats = take(fused_one ? row_splits * 16 : 0);
  pl.off_pending = take(pl.one_launch ? row_splits * 4 : 0);
  pl.off_best = take(fused_two ? rows * 8 : 0);
  pl.off_tail = take(fused_two ? 8 : 0);
  off = (off + 255) & ~(size_t)255;
  pl.off_count = take(pl.one_launch || fused_h2o ? rows * kCountStride * 4 : 0);
  pl.total = (off + 255) & ~(size_t)255;
  return pl;
}

DecodeCounters counters_of(const DecodeParams& p) {
  return {p.row_count, p.scratch_splits, (unsigned long long*)p.part_ml, (int64_t)p.B * p.Hq * p.num_splits};
}

}  // namespace

size_t sdpa_decode_workspace(const kvx_sdpa_args& a, bool fused_h2o) { return make_plan(a, fused_h2o).total; }

void set_decode_tuning(int resident, int spin_limit, int poll_sleep) {
  Tuning& t = tuning();
  t.resident = resident < 0 ? t.env_resident : (resident != 0);
  t.spin_limit = spin_limit < 0 ? t.env_spin : clampi(spin_limit, 0, kSpinMax);
  t.poll_sleep = poll_sleep < 0 ? t.env_sleep : clampi(poll_sleep, 0, kSleepMax);
}

void decode_wait(int& spin_limit, int& poll_sleep) {
  spin_limit = tuning().spin_limit.load();
  poll_sleep = tuning().poll_sleep.load();
}

namespace {
int decode_params(DecodeParams& p, const kvx_sdpa_args& a, const kvx_h2o_args* hh, const Plan& pl) {
  KVX_REQUIRE(a.workspace && a.workspace_bytes >= pl.total, KVX_ERR_WORKSPACE,
              "kvx_sdpa_decode: workspace of %zu bytes needed, %zu given", pl.total, a.workspace_bytes);
  const int64_t es = kv_is_plain(a.kv_dtype) ? 2 : 1;
  KVX_REQUIRE((int64_t)a.kv_len * a.k_stride_t * es < (1ll << 32) && (int64_t)a.kv_len * a.v_stride_t * es < (1ll << 32), KVX_ERR_UNSUPPORTED,
              "kvx_sdpa_decode: one (batch, head) row set of K or V must span less than 4 GiB (kv_len %d, slot strides %lld / %lld)",
              a.kv_len, (long long)a.k_stride_t, (long long)a.v_stride_t);
  char* ws = (char*)a.workspace;
  p.q = (const uint16_t*)a.q;
  p.k = a.k;
  p.v = a.v;
  p.k_scale = a.k_scale; p.k_zp = a.k_zp; p.v_scale = a.v_scale; p.v_zp = a.v_zp;
  p.o = (uint16_t*)a.o;
  p.lse_out = a.lse;
  p.w = a.w;
  p.logits = (a.w || hh) ? (float*)(ws + pl.off_logits) : nullptr;
  p.part_o = (float*)(ws + pl.off_part_o);
  p.part_ml = (float*)(ws + pl.off_part_ml);
  const bool two = hh && !pl.one_launch;
  p.best = two ? (unsigned long long*)(ws + pl.off_best) : nullptr;
  p.tail_count = two ? (uint32_t*)(ws + pl.off_tail) : nullptr;
  p.row_count = (uint32_t*)(ws + pl.off_count);
  p.part_best = (unsigned long long*)(ws + pl.off_part_best);
  p.part_vn = (float*)(ws + pl.off_part_vn);
  p.part_stats = (float*)(ws + pl.off_part_stats);
  p.split_pending = (uint32_t*)(ws + pl.off_pending);
  p.scratch_splits = a.decode_scratch_splits;
  p.resident = pl.resident;
  p.one_launch = pl.one_launch;
  p.spin_limit = tuning().spin_limit.load();
  p.poll_sleep = tuning().poll_sleep.load();
  p.B = a.B; p.Hq = a.Hq; p.Hkv = a.Hkv; p.kv_len = a.kv_len; p.Tpad = pl.Tpad;
  p.Gr = a.Hq / a.Hkv;
  KVX_REQUIRE(p.Gr <= 16, KVX_ERR_UNSUPPORTED, "kvx_sdpa_decode: more than 16 query heads per KV head (%d)", p.Gr);
  p.qs_vec = (((uintptr_t)a.k_scale | (uintptr_t)a.k_zp | (uintptr_t)a.v_scale | (uintptr_t)a.v_zp) & 15) == 0 && a.qs_stride_b % 4 == 0 && a.qs_stride_h % 4 == 0;
  p.num_splits = pl.num_splits; p.keys_per_split = pl.keys_per_split;
  p.share = (p.Gr * (a.D / 2) + pl.num_splits - 1) / pl.num_splits;
  p.scores = hh != nullptr;
  p.positions = hh && hh->normalize;
  p.lj = pl.num_splits <= 4 ? 0 : pl.num_splits <= 8 ? 1 : pl.num_splits <= 16 ? 2 : pl.num_splits <= 32 ? 3 : 4;
  p.inv_g = 1.0f / (float)p.Gr;
  p.c = a.sm_scale * kLog2e;
  p.q_sb = a.q_stride_b; p.q_sh = a.q_stride_h;
  p.k_sb = a.k_stride_b; p.k_sh = a.k_stride_h; p.k_st = a.k_stride_t;
  p.v_sb = a.v_stride_b; p.v_sh = a.v_stride_h; p.v_st = a.v_stride_t;
  p.o_sb = a.o_stride_b; p.o_sh = a.o_stride_h;
  p.qs_sb = a.qs_stride_b; p.qs_sh = a.qs_stride_h;
  return KVX_OK;
}

// The reset of counters and of the splits' maxima and sums (unless `counters_clear`: the slot write before did it, or there is a single split), then the kernels.
int launch_split(const DecodeParams& p, int D, int G, int kv, const kvx_h2o_args* hh, bool counters_clear, hipStream_t st) {
  const int rows = p.B * p.Hkv;
  const bool counts = p.one_launch ? p.num_splits > 1 && !counters_clear : hh != nullptr;
  if (counts || (p.scratch_splits && !counters_clear)) {
    // splits that take the scratch route by plan (the resident form switched off or too long for the LDS) count from the start
    const uint32_t by_plan = (p.logits && !p.resident) ? (uint32_t)(rows * p.num_splits) : 0u;
    DecodeCounters c = counters_of(p);
    if (!counts) c.rows = nullptr;
    if (!counts || !p.one_launch) c.pairs = 0;
    const int64_t lanes = max((int64_t)rows, c.pairs / 4);
    hipLaunchKernelGGL(decode_init_kernel, dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, st, c, p.best, p.tail_count, rows, by_plan);
    KVX_HIP(hipGetLastError());
  }
  if (D == 128) return launch_decode_128(p, G, kv, hh, st);
  if (D == 64) return launch_decode_64(p, G, kv, hh, st);
  if (D == 256) return launch_decode_256(p, G, kv, hh, st);
  return set_error(KVX_ERR_UNSUPPORTED, "kvx_sdpa_decode: head size %d not in {64, 128, 256}", D);
}
}  // namespace

int launch_sdpa_decode(const kvx_sdpa_args& a, const kvx_h2o_args* hh, hipStream_t st) {
  const Plan pl = make_plan(a, hh != nullptr);
  DecodeParams p;
  const int rc = decode_params(p, a, hh, pl);
  return rc != KVX_OK ? rc : launch_split(p, a.D, pl.G, a.kv_dtype, hh, false, st);
}

// ---- a whole cache step of one token: the slot write clears the counters, the split kernel does the rest -----------

static bool step_is_variant(const kvx_h2o_args& h) { return h.v_norm || h.q_errors; }
static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

size_t decode_step_workspace(const kvx_sdpa_args& a, const kvx_h2o_args& h) {
  const Plan pl = make_plan(a, true);
  if (pl.one_launch) return pl.total;
  // logits through the scratch by plan: the calls this one stands for, one after the other
  if (!step_is_variant(h)) return align256(h2o_workspace(h)) + pl.total;
  kvx_sdpa_args aw = a;
  aw.w = (float*)a.k;  // any pointer: score-sums are wanted
  return align256(h2o_workspace(h)) + align256((size_t)a.B * a.Hkv * a.kv_len * 4) + make_plan(aw, false).total;
}

int launch_decode_step(const kvx_cache_write_args& w, const kvx_sdpa_args& a, const kvx_h2o_args& h, hipStream_t st) {
  const Plan pl = make_plan(a, true);
  KVX_REQUIRE(a.workspace && a.workspace_bytes >= decode_step_workspace(a, h), KVX_ERR_WORKSPACE,
              "kvx_h2o_decode_step: workspace of %zu bytes needed, %zu given", decode_step_workspace(a, h), a.workspace_bytes);
  if (!pl.one_launch) {
    int rc = launch_cache_write(w, nullptr, st);
    if (rc != KVX_OK) return rc;
    kvx_sdpa_args a2 = a;
    kvx_h2o_args h2 = h;
    char* ws = (char*)a.workspace;
    h2.workspace = ws;
    h2.workspace_bytes = align256(h2o_workspace(h));
    ws += h2.workspace_bytes;
    if (step_is_variant(h)) {
      a2.w = (float*)ws;
      h2.w = a2.w;
      ws += align256((size_t)a.B * a.Hkv * a.kv_len * 4);
    }
    a2.workspace = ws;
    a2.workspace_bytes = (size_t)((char*)a.workspace + a.workspace_bytes - ws);
    rc = launch_sdpa_decode(a2, step_is_variant(h) ? nullptr : &h2, st);
    return rc != KVX_OK || !step_is_variant(h) ? rc : launch_h2o_update_select(h2, st);
  }
  DecodeParams p;
  int rc = decode_params(p, a, &h, pl);
  if (rc != KVX_OK) return rc;
  const DecodeCounters counters = counters_of(p);
  rc = launch_cache_write(w, &counters, st);
  if (rc != KVX_OK) return rc;
  rc = launch_split(p, a.D, pl.G, a.kv_dtype, &h, true, st);
  if (rc != KVX_OK || !h.q_errors) return rc;
  return launch_select_one(h, p.part_stats, p.num_splits, p.row_count + kSelected, p.part_best, st);
}

}  // namespace kvx
