// RMS normalisation of rows, and the per-head query/key normalisation fused with the rotary position
// encoding, for gfx950 (both HBM-bound, one pass).
//
// Reference behaviour:
//   RMSNorm.forward, keys_values/model.py:870-878: x32 = float(x); n = |x32|_2 / sqrt(size);
//     y = (x32 / (n + eps)) * weight, cast to the input type. eps is added to the norm, not under the
//     root, and the division happens before the multiplication by the weight.
//   CausalSelfAttention.forward, keys_values/model.py:733-775: q and k are normalised per head over
//     head_size (norm_q / norm_k), cast back to bf16, then rotated (apply_rope,
//     keys_values/pos_encoding.py:34-44 -> y = x * cos + cat(-x2, x1) * sin in fp32, half-split
//     convention, keys_values/fused/fused_rope.py:57-87,198-200) and cast to bf16 again.
// The fused kernel keeps both casts, so it returns what the two separate steps return. It works in
// place on the output of the QKV projection, (B, num, (Hq + 2 Hkv) * D): the value heads are left as
// they are and no transposed copies are made (the attention and cache kernels take strides).
#include <type_traits>

#include "kvx_common.h"

namespace kvx {
namespace {

constexpr int NT = 256;

// These kernels move two or four bytes a value, and what bounded them was the vector ALU: an IEEE division takes a dozen instructions and a 64-bit index
// division about a hundred. Values of a row are divided by the row's norm, so one division serves them: with r = RN(1 / b), q = RN(a r) and
// the remainder q b - a, exact in a fused multiply-add, q - (q b - a) r is RN(a / b) (Markstein, "Computation of elementary functions on the IBM
// RISC System/6000 processor", 1990) while nothing over- or underflows: by norms of 2^-40 to 2^40, of values from 2^-85 (the quotient is
// above 2^-126, the remainder's last bit above 2^-149) to the norm times sqrt(dim). Of smaller ones the last bit of the quotient may differ. The remainder is formed as q b - a and not as a - q b, so that a zero keeps its sign. Other norms (zero rows with eps = 0,
// infinities, NaN) are divided by as they are.
struct Divisor {
  float b, r;
  bool plain;
  __device__ __forceinline__ explicit Divisor(float x) : b(x), r(1.0f / x), plain(x > 0x1p-40f && x < 0x1p40f) {}
  __device__ __forceinline__ float under(float a) const {
    const float q = a * r;
    return fmaf(fmaf(q, b, -a), -r, q);
  }
};
// v of one lane, 8 values, divided by the norm, times the weights
template <typename Store>
__device__ __forceinline__ void normalised(const float (&x)[8], const Divisor& d, const f32x4_t& w0, const f32x4_t& w1, Store store) {
  float y[8];
  if (__all(d.plain)) {
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = d.under(x[e]) * (e < 4 ? w0[e] : w1[e - 4]);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = (x[e] / d.b) * (e < 4 ? w0[e] : w1[e - 4]);
  }
  store(y);
}
__device__ __forceinline__ void unpack(const u32x4_t& v, float (&x)[8]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    x[2 * e] = bf16_lo(v[e]);
    x[2 * e + 1] = bf16_hi(v[e]);
  }
}
__device__ __forceinline__ u32x4_t packed(const float (&y)[8]) {
  return u32x4_t{pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3]), pack_bf16(y[4], y[5]), pack_bf16(y[6], y[7])};
}

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off, 64);
  return x;
}

// Sum over the WPR wavefronts that share a row (more than one: through LDS, added in wavefront order).
template <int WPR>
__device__ __forceinline__ float row_total(float ss) {
  ss = wave_sum(ss);
  if constexpr (WPR > 1) {
    __shared__ float part[WPR];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = part[0];
#pragma unroll
    for (int i = 1; i < WPR; ++i) ss += part[i];
  }
  return ss;
}

// Threads of a workgroup: one row of several wavefronts, or rows of one each. The kernels of the latter are compiled for 512, which schedules the sum's loads 2 %
// better in the mean and the plain norm's 2 % worse.
constexpr int norm_threads(int WPR) { return WPR > 1 ? 64 * WPR : NT; }
constexpr int norm_bound(int WPR) { return WPR > 1 ? 64 * WPR : 512; }

// WPR wavefronts a row; a lane holds up to MAXC chunks of 8 elements (dim <= 64 * WPR * 8 * MAXC).
// Few long rows (a 1024-token chunk of hidden states) take a workgroup per row (by_row_length).
template <int MAXC, int WPR>
__global__ __launch_bounds__(norm_bound(WPR)) void rmsnorm_rows_kernel(const uint16_t* __restrict__ x, int64_t x_rs, uint16_t* __restrict__ out,
                                                          int64_t o_rs, const float* __restrict__ weight, int64_t rows, int dim,
                                                          float eps, float factor) {
  constexpr int TPR = 64 * WPR;  // threads per row
  const int lane = threadIdx.x % TPR;
  const int64_t row = (int64_t)blockIdx.x * (norm_threads(WPR) / TPR) + threadIdx.x / TPR;
  if (row >= rows) return;  // uniform over the threads of a row (and over the workgroup where it shares one)
  const int nchunks = dim / 8;
  const uint16_t* xr = x + row * x_rs;
  u32x4_t v[MAXC];
  float ss = 0.0f;
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int ch = lane + TPR * c;
    v[c] = u32x4_t{0, 0, 0, 0};
    if (ch < nchunks) v[c] = *(const u32x4_t*)(xr + ch * 8);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = bf16_lo(v[c][e]), b = bf16_hi(v[c][e]);
      ss += a * a;
      ss += b * b;
    }
  }
  ss = row_total<WPR>(ss);
  const Divisor denom(sqrtf(ss) * factor + eps);
  uint16_t* orow = out + row * o_rs;
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int ch = lane + TPR * c;
    if (ch >= nchunks) break;
    const f32x4_t w0 = *(const f32x4_t*)(weight + ch * 8);
    const f32x4_t w1 = *(const f32x4_t*)(weight + ch * 8 + 4);
    float f[8];
    unpack(v[c], f);
    normalised(f, denom, w0, w1, [&](const float (&y)[8]) { *(u32x4_t*)(orow + ch * 8) = packed(y); });
  }
}

// x_out = bf16(x + delta) and out = RMSNorm(x_out) in one pass: the residual add of a block fused with
// the normalisation that follows it (keys_values/model.py:560-584: x = attention_output + x, then
// norm_2(x); x = mlp_output + x, then the next block's norm_1). The sum is rounded to bf16 before it is
// normalised, as the two separate steps do. In place is allowed (x_out == x).
template <int MAXC, int WPR>
__global__ __launch_bounds__(norm_bound(WPR)) void add_rmsnorm_rows_kernel(const uint16_t* x, int64_t x_rs, const uint16_t* __restrict__ delta,
                                                              int64_t d_rs, uint16_t* x_out, int64_t xo_rs,
                                                              uint16_t* __restrict__ out, int64_t o_rs, const float* __restrict__ weight,
                                                              int64_t rows, int dim, float eps, float factor) {
  constexpr int TPR = 64 * WPR;
  const int lane = threadIdx.x % TPR;
  const int64_t row = (int64_t)blockIdx.x * (norm_threads(WPR) / TPR) + threadIdx.x / TPR;
  if (row >= rows) return;
  const int nchunks = dim / 8;
  u32x4_t v[MAXC];
  float ss = 0.0f;
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int ch = lane + TPR * c;
    v[c] = u32x4_t{0, 0, 0, 0};
    if (ch < nchunks) {
      const u32x4_t a = *(const u32x4_t*)(x + row * x_rs + ch * 8);
      const u32x4_t b = *(const u32x4_t*)(delta + row * d_rs + ch * 8);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[c][e] = pack_bf16(bf16_lo(a[e]) + bf16_lo(b[e]), bf16_hi(a[e]) + bf16_hi(b[e]));
      *(u32x4_t*)(x_out + row * xo_rs + ch * 8) = v[c];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = bf16_lo(v[c][e]), b = bf16_hi(v[c][e]);
      ss += a * a;
      ss += b * b;
    }
  }
  ss = row_total<WPR>(ss);
  const Divisor denom(sqrtf(ss) * factor + eps);
  uint16_t* orow = out + row * o_rs;
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int ch = lane + TPR * c;
    if (ch >= nchunks) break;
    const f32x4_t w0 = *(const f32x4_t*)(weight + ch * 8);
    const f32x4_t w1 = *(const f32x4_t*)(weight + ch * 8 + 4);
    float f[8];
    unpack(v[c], f);
    normalised(f, denom, w0, w1, [&](const float (&y)[8]) { *(u32x4_t*)(orow + ch * 8) = packed(y); });
  }
}

// out[r, j] = bf16( bf16(silu(g[r, j])) * u[r, j] ), g = gate_up[r, j], u = gate_up[r, dim + j]: the
// gated activation of LLaMAMLP (proj(silu(fc_1 x) * fc_2 x)) on the output of one GEMM over the stacked
// fc_1 / fc_2 weights. silu is x / (1 + exp(-x)) in fp32, rounded to bf16 before the product, as the
// two separate tensor operations round.
// exp(-x) is 2^h (1 + l ln 2) with h + l = -x log2(e), h rounded; the quotient as in Divisor, of a reciprocal that is an ulp off. Values below -80, whose
// exponential is near the type's end, and NaN take the divisions. Of all 16-bit gates the error is 0.069 of the last of 24 bits in the mean and 1.77 at most, that of
// expf and a division 0.068 and 1.75, and the 16 bits that are kept are the same. With expf, a division each and 64-bit indexes the kernel was bound by the vector ALU:
// 4096 / 1024 rows of 9728 values 42.2 -> 39.3 and 13.3 -> 12.1 us.
__device__ __forceinline__ float silu(float x) {
  constexpr float L2E = 1.4426950408889634f, L2E_LOW = (float)(1.4426950408889634 - (double)L2E), LN2 = 0.6931471805599453f;
  const float h = x * -L2E, l = fmaf(x, -L2E, -h) + x * -L2E_LOW;
  const float p = fast_exp2(h), d = 1.0f + fmaf(p, l * LN2, p);
  const float r = __builtin_amdgcn_rcpf(d), q = x * r;
  return fmaf(fmaf(q, d, -x), -r, q);
}
__global__ __launch_bounds__(NT) void swiglu_rows_kernel(const uint16_t* __restrict__ gate_up, int64_t g_rs, uint16_t* __restrict__ out,
                                                         int64_t o_rs, uint32_t rows, int dim) {
  const uint32_t cpr = dim / 8, gid = blockIdx.x * NT + threadIdx.x;
  const int64_t r = gid / cpr;
  const int c = gid % cpr;
  if (r >= rows) return;
  const u32x4_t g = *(const u32x4_t*)(gate_up + r * g_rs + c * 8);
  const u32x4_t u = *(const u32x4_t*)(gate_up + r * g_rs + dim + c * 8);
  float x[8];
  unpack(g, x);
  bool plain = true;
#pragma unroll
  for (int e = 0; e < 8; ++e) plain = plain && x[e] > -80.0f && x[e] < 0x1p100f;
  u32x4_t act;
  if (__all(plain)) {
#pragma unroll
    for (int e = 0; e < 4; ++e) act[e] = pack_bf16(silu(x[2 * e]), silu(x[2 * e + 1]));
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) act[e] = pack_bf16(x[2 * e] / (1.0f + expf(-x[2 * e])), x[2 * e + 1] / (1.0f + expf(-x[2 * e + 1])));
  }
  u32x4_t o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = pack_bf16(bf16_lo(act[e]) * bf16_lo(u[e]), bf16_hi(act[e]) * bf16_hi(u[e]));
  *(u32x4_t*)(out + r * o_rs + c * 8) = o;
}

// Sum of the squares of half a row, four values a lane, for all LPR lanes: runs of eight values one after the other, then the runs in pairs, which is the order of
// lanes that hold eight values in a row.
template <int LPR>
__device__ __forceinline__ float half_sum(float a, float b, float c, float d) {
  auto of_even = [](float x) { return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0xA0, 0xf, 0xf, true)); };  // quad_perm [0,0,2,2]
  auto of_odd = [](float x) { return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0xF5, 0xf, 0xf, true)); };   // quad_perm [1,1,3,3]
  const float aa = a * a, bb = b * b, cc = c * c, dd = d * d;
  float ss = of_odd(of_even(aa + bb + cc + dd) + aa + bb + cc + dd);
#pragma unroll
  for (int off = 2; off < LPR; off <<= 1) ss += __shfl_xor(ss, off, 64);
  return ss;
}

// A workgroup, or several (grid y), per token: the rows are its query heads, then its key heads; LPR = D / 8 lanes a row hold four values of either half of it, so
// a value and the one it is rotated with are in the same lane; the angles and weights of a lane are the same for all its rows. `rows` of a workgroup at a time (each of U), every
// `stride` heads. With a row's values in a stretch a lane, partners through LDS and a row's place by 64-bit divisions: 22.4 -> 16.8 us for 40 heads of 128 of 4096 tokens,
// 8.0 -> 5.8 of 1024.
template <int D, int U>  // U: rows of a lane in flight
__global__ __launch_bounds__(512) void qk_norm_rope_kernel(uint16_t* __restrict__ qkv, int64_t sb, int64_t st, int num, int Hq,
                                                          int Hkv, const float* __restrict__ qw, const float* __restrict__ kw,
                                                          float eps, float factor, const float* __restrict__ cos_t,
                                                          const float* __restrict__ sin_t, int input_pos, int rows, int stride) {
  constexpr int LPR = D / 8;
  constexpr int HALF = D / 2;
  const int col = threadIdx.x % LPR, first = threadIdx.x / LPR;
  const int heads = Hq + Hkv;
  const int b = blockIdx.x / num, t = blockIdx.x - b * num;
  uint16_t* p = qkv + b * sb + (int64_t)t * st + col * 4;
  const f32x4_t cv = *(const f32x4_t*)(cos_t + (int64_t)(input_pos + t) * HALF + col * 4);
  const f32x4_t sv = *(const f32x4_t*)(sin_t + (int64_t)(input_pos + t) * HALF + col * 4);
  for (int begin = blockIdx.y * U * rows; begin < heads; begin += stride) {
    u32x2_t lo[U], hi[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int head = min(begin + i * rows + first, heads - 1);
      lo[i] = *(const u32x2_t*)(p + head * D);
      hi[i] = *(const u32x2_t*)(p + head * D + HALF);
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int head = begin + i * rows + first;
      float y[8];
      unpack(u32x4_t{lo[i][0], lo[i][1], hi[i][0], hi[i][1]}, y);
      if (qw) {  // either both weights are given or none
        const float ss = half_sum<LPR>(y[0], y[1], y[2], y[3]) + half_sum<LPR>(y[4], y[5], y[6], y[7]);
        const float* w = (head < Hq ? qw : kw) + col * 4;
        normalised(y, Divisor(sqrtf(ss) * factor + eps), *(const f32x4_t*)w, *(const f32x4_t*)(w + HALF), [&](const float (&z)[8]) {
          // the reference casts the normalised head back to bf16 before it is rotated
          unpack(packed(z), y);
        });
      }
      // rotation: the first half gets -x2, the second +x1
      float x[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = y[e] * cv[e] + -y[e + 4] * sv[e];
        x[e + 4] = y[e + 4] * cv[e] + y[e] * sv[e];
      }
      const u32x4_t o = packed(x);
      if (head < heads) {
        *(u32x2_t*)(p + head * D) = u32x2_t{o[0], o[1]};
        *(u32x2_t*)(p + head * D + HALF) = u32x2_t{o[2], o[3]};
      }
    }
  }
}

// Rows of at least 2048 values take a workgroup each where they are too few to fill the chip with a wavefront each: four wavefronts, and five to eight above
// 4096 values, so that a lane holds two chunks at most. A wavefront for each chunk of a lane, counted at run time, held fewer rows in flight on a unit, and the count came from
// memory. us, norm of 1024 rows of 2560 4.6 that way, 3.6 now (with a division a value and four wavefronts 4.1), of 4096 x 4096 15.8, 12.3 (13.7), of 16384 x 2560 31.5, 25.3 (27.7);
// sum and norm of 1024 x 2560 5.4, 5.0 (5.7), 1024 x 4096 7.7, 5.9 (6.7), 1024 x 8192 10.2, 9.6 (11.6). Beyond the last-level cache eight wavefronts win from about 3600 values on: sums of
// 16384 x 4096 95.7 with four, 91.3, of 12000 x 3840 60.6, 58.9, but of 10000 x 4096 46.9, 47.7 and of 16384 x 3072 65.5, 67.2. Above 4096 sums take no wavefront that half a row
// leaves idle (8000 x 7168: seven 71, eight 74.4), norms alone eight (16384 x 7168: 88, 84). Rows of
// 2048 take the kernel of two chunks as well, at the same bits: 1024 rows 3.3, with the second chunk left out 3.9. `tensors`: read and written.
// `launch(chunks a lane, wavefronts a row, grid)`
template <typename Launch>
void by_row_length(int64_t rows, int dim, int tensors, Launch launch) {
  constexpr std::integral_constant<int, 1> I1{};
  constexpr std::integral_constant<int, 2> I2{};
  constexpr std::integral_constant<int, 4> I4{};
  if (dim >= 2048 && rows <= 16384) {
    if (dim <= 3584 || (dim <= 4096 && rows * dim * 2 * tensors <= (336ll << 20))) launch(I2, I4, (unsigned)rows);
    else if (dim <= 4096 || dim > 7168 || tensors == 2) launch(I2, std::integral_constant<int, 8>{}, (unsigned)rows);
    else if (dim <= 5120) launch(I2, std::integral_constant<int, 5>{}, (unsigned)rows);
    else if (dim <= 6144) launch(I2, std::integral_constant<int, 6>{}, (unsigned)rows);
    else launch(I2, std::integral_constant<int, 7>{}, (unsigned)rows);
  } else if (dim <= 64 * 8 * 4) {
    launch(I4, I1, (unsigned)((rows + NT / 64 - 1) / (NT / 64)));
  } else {
    launch(std::integral_constant<int, 16>{}, I1, (unsigned)((rows + NT / 64 - 1) / (NT / 64)));
  }
}

}  // namespace

int launch_rmsnorm_rows(const void* x, int64_t x_rs, void* out, int64_t o_rs, const float* weight, int64_t rows, int dim, float eps,
                        hipStream_t st) {
  if (rows == 0) return KVX_OK;
  const float factor = 1.0f / sqrtf((float)dim);
  by_row_length(rows, dim, 2, [&](auto chunks, auto waves, unsigned grid) {
    constexpr int MAXC = decltype(chunks)::value, WPR = decltype(waves)::value;
    hipLaunchKernelGGL((rmsnorm_rows_kernel<MAXC, WPR>), dim3(grid), dim3(norm_threads(WPR)), 0, st, (const uint16_t*)x, x_rs,
                       (uint16_t*)out, o_rs, weight, rows, dim, eps, factor);
  });
  KVX_HIP(hipGetLastError());
  return KVX_OK;
}

int launch_add_rmsnorm_rows(const void* x, int64_t x_rs, const void* delta, int64_t d_rs, void* x_out, int64_t xo_rs, void* out,
                            int64_t o_rs, const float* weight, int64_t rows, int dim, float eps, hipStream_t st) {
  if (rows == 0) return KVX_OK;
  const float factor = 1.0f / sqrtf((float)dim);
  by_row_length(rows, dim, 4, [&](auto chunks, auto waves, unsigned grid) {
    constexpr int MAXC = decltype(chunks)::value, WPR = decltype(waves)::value;
    hipLaunchKernelGGL((add_rmsnorm_rows_kernel<MAXC, WPR>), dim3(grid), dim3(norm_threads(WPR)), 0, st, (const uint16_t*)x, x_rs,
                       (const uint16_t*)delta, d_rs, (uint16_t*)x_out, xo_rs, (uint16_t*)out, o_rs, weight, rows, dim, eps, factor);
  });
  KVX_HIP(hipGetLastError());
  return KVX_OK;
}

int launch_swiglu_rows(const void* gate_up, int64_t g_rs, void* out, int64_t o_rs, int64_t rows, int dim, hipStream_t st) {
  const int64_t at_once = (1u << 31) / (dim / 8);  // rows whose chunks have 32-bit indexes
  for (int64_t done = 0; done < rows; done += at_once) {
    const int64_t n = rows - done < at_once ? rows - done : at_once;
    hipLaunchKernelGGL(swiglu_rows_kernel, dim3((unsigned)((n * (dim / 8) + NT - 1) / NT)), dim3(NT), 0, st, (const uint16_t*)gate_up + done * g_rs, g_rs,
                       (uint16_t*)out + done * o_rs, o_rs, (uint32_t)n, dim);
    KVX_HIP(hipGetLastError());
  }
  return KVX_OK;
}

int launch_qk_norm_rope(void* qkv, int64_t sb, int64_t stt, int B, int num, int Hq, int Hkv, int D, const float* qw, const float* kw,
                        float eps, const float* cos_t, const float* sin_t, int input_pos, hipStream_t st) {
  if (B == 0 || num == 0 || Hq + Hkv == 0) return KVX_OK;
  const float factor = 1.0f / sqrtf((float)D);
  const int lanes = (Hq + Hkv) * (D / 8), lpr = D / 8;
  const int at_once = max(1, (1 << 22) / num);  // batch elements whose threads a grid can count
  const int64_t tokens = (int64_t)min(at_once, B) * num;
  // A token's rows over several workgroups where few tokens leave units idle or its rows are many; over one, two rows a lane, where up to 640 lanes of many
  // tokens would read the angles again. us, one / several: 16 tokens of 72 heads of 256 5.8 / 2.6, of 40 of 128 3.2 / 2.5, 1024 of 72 of 128 10.7 / 8.6; 4096 of 40 of
  // 64 9.8 / 11.2, of 10 of 256 10.0 / 11.4, 1024 of 40 of 128 5.8 / 6.1. (A workgroup a token for all: 16 of 72 of 256 6.1, as lanes of rows in a
  // stretch 3.2.)
  const int parts = lanes > 2 * NT + 128 || tokens <= 2 * num_cus() ? min((lanes + NT - 1) / NT, 65535) : 1;
  const int rows = parts > 1 || lanes <= NT ? 1 : 2;  // of a lane
  const int threads = parts > 1 ? NT : (lanes / rows + 63) / 64 * 64;
  auto launch = [&](auto kernel) {
    for (int done = 0; done < B; done += at_once)
      hipLaunchKernelGGL(kernel, dim3((unsigned)(min(at_once, B - done) * num), parts), dim3(threads), 0, st, (uint16_t*)qkv + done * sb, sb, stt, num, Hq, Hkv, qw, kw, eps,
                         factor, cos_t, sin_t, input_pos, threads / lpr, parts * rows * (threads / lpr));
  };
  auto launch_d = [&](auto d_tag) {
    constexpr int HEAD = decltype(d_tag)::value;
    if (rows == 1) launch(qk_norm_rope_kernel<HEAD, 1>);
    else launch(qk_norm_rope_kernel<HEAD, 2>);
  };
  if (D == 256) launch_d(std::integral_constant<int, 256>{});
  else if (D == 128) launch_d(std::integral_constant<int, 128>{});
  else launch_d(std::integral_constant<int, 64>{});
  KVX_HIP(hipGetLastError());
  return KVX_OK;
}

}  // namespace kvx
