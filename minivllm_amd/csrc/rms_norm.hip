// mvllm_add_rms_norm: the decoder layer's residual add + RMSNorm in one launch.
// Reference: LayerNorm.forward / residual_rms_forward / rms_forward, src/myvllm/layers/layernorm.py:9-28
//   x = x + residual                                   (in the element type: the sum is rounded to it)
//   out = x / sqrt(mean(x^2) + eps) * gamma, residual_out = x
// as called twice per layer and once after the last layer (src/myvllm/models/qwen3.py:197-212, 306-312).
// The norm is computed in fp32 from the rounded sum with separate multiplies and adds (no contraction), a
// correctly rounded square root and the quotient x / denominator taken with one correction step from the
// correctly rounded reciprocal (SharedDivisor); only the order of the sum of squares is free.
//
// WAVES waves per row; thread l of them holds elements [8 (l + 64 WAVES c), +8) for chunks c = 0 .. CHUNKS-1 in registers, so the
// row is read once and written once (16-byte accesses).  Up to 1024 numbers a row takes one wave; longer ones four, because a wave with
// 32 numbers or more per lane to take through the norm is what few rows wait for, and holds too many registers to have enough rows
// under way where there are many (us with one wave and with four: 61 rows of 4096 6.6 / 3.1, 1024 rows 8.8 / 6.5, 8192 rows 44.7 / 39.6;
// 8192 rows of 8192 135 / 103 = 5.2 TB/s).  Many rows just above 1024: see kManyRows.
#include "common.h"

#pragma clang fp contract(off)

namespace mvllm {

template <typename T> struct Row8;
template <> struct Row8<float> {
  static __device__ __forceinline__ void load(const float* p, float (&x)[8]) {
    const float4 a = *reinterpret_cast<const float4*>(p);
    const float4 b = *reinterpret_cast<const float4*>(p + 4);
    x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
    x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
  }
  static __device__ __forceinline__ void store(float* p, const float (&x)[8]) {
    *reinterpret_cast<float4*>(p) = make_float4(x[0], x[1], x[2], x[3]);
    *reinterpret_cast<float4*>(p + 4) = make_float4(x[4], x[5], x[6], x[7]);
  }
};
template <typename T16> struct Row8 {
  static __device__ __forceinline__ void load(const T16* p, float (&x)[8]) {
    const uint4 w = *reinterpret_cast<const uint4*>(p);
    x[0] = lo_to_float<T16>(w.x); x[1] = hi_to_float<T16>(w.x);
    x[2] = lo_to_float<T16>(w.y); x[3] = hi_to_float<T16>(w.y);
    x[4] = lo_to_float<T16>(w.z); x[5] = hi_to_float<T16>(w.z);
    x[6] = lo_to_float<T16>(w.w); x[7] = hi_to_float<T16>(w.w);
  }
  static __device__ __forceinline__ void store(T16* p, const float (&x)[8]) {
    T16 o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = from_float<T16>(x[e]);
    *reinterpret_cast<uint4*>(p) = *reinterpret_cast<const uint4*>(o);
  }
};

constexpr int kNormThreads = 256;   // 4 rows per workgroup

template <typename T, int CHUNKS, int WAVES>
__global__ __launch_bounds__(kNormThreads) void add_rms_norm_kernel(
    T* __restrict__ out, T* __restrict__ residual_out, const T* __restrict__ x, const T* __restrict__ residual,
    const float* __restrict__ gamma, float eps, int64_t rows, int hidden, int64_t x_stride, int64_t res_stride) {
  constexpr int kRows = kNormThreads / 64 / WAVES;
  __shared__ float part[WAVES > 1 ? kNormThreads / 64 : 1];
  const int lane = threadIdx.x & (64 * WAVES - 1);
  const int64_t row = (int64_t)blockIdx.x * kRows + threadIdx.x / (64 * WAVES);
  if (row >= rows) return;                            // (WAVES > 1: one row per workgroup, so all of it)
  static_assert(WAVES == 1 || kRows == 1, "the workgroup's barrier is the row's");
  const T* xp = x + row * x_stride;
  float v[CHUNKS][8];
  // gamma does not depend on the row: it is fetched together with the row instead of after the
  // reduction, which takes one memory latency out of a kernel that is all latency at decode batch sizes
  float gam[CHUNKS][8];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int e0 = 8 * (lane + 64 * WAVES * c);
    if (e0 < hidden) {
      Row8<T>::load(xp + e0, v[c]);
      Row8<float>::load(gamma + e0, gam[c]);
      if (residual) {
        float r[8];
        Row8<T>::load(residual + row * res_stride + e0, r);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[c][e] = to_float(from_float<T>(v[c][e] + r[e]));   // the sum lives in T
      }
      if (residual_out) Row8<T>::store(residual_out + row * (int64_t)hidden + e0, v[c]);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = ss + v[c][e] * v[c][e];
    }
  }
  ss = four_rows_sum(row16_sum(ss));
  if constexpr (WAVES > 1) {
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = part[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) ss = ss + part[w];
  }
  const SharedDivisor denom(sqrtf(ss / (float)hidden + eps));
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int e0 = 8 * (lane + 64 * WAVES * c);
    if (e0 < hidden) {
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = denom.divide(v[c][e]) * gam[c][e];
      Row8<T>::store(out + row * (int64_t)hidden + e0, y);
    }
  }
}

// ... but not where half the threads of four waves would have no element and rows enough are there to fill the chip: a row just above 1024
// numbers stays in one wave (with a residual twice the loads are under way, and fewer of them idle).  us in four and in one, 3072 /
// 8192 / 65536 rows: of 1032 numbers 5.2 / 9.4 / 55.7 and 5.1 / 8.2 / 45.6, of 1280 5.2 / 9.5 / 69.8 and 4.9 / 8.5 / 61.8, of 1536 5.4 / 9.9 / 74 and
// 5.2 / 9.1 / 72 but 16.6 and 16.7 at 16384; with a residual 1032 6.9 / 14.2 / 110 and 6.7 / 13.5 / 110, 1152 6.9 / 13.7 / 109 and 6.8 / 13.9 / 111.
// 2048 rows of 1280 in four 4.3, in one 4.5.
constexpr int64_t kManyRows = 3072;

template <typename T>
static int launch_norm(void* out, void* residual_out, const void* x, const void* residual, const float* gamma, float eps,
                       int64_t rows, int hidden, int64_t x_stride, int64_t res_stride, hipStream_t s) {
  const int chunks = (hidden + 511) / 512;
  const bool one_wave = chunks <= 2 || (rows >= kManyRows && hidden <= (residual ? 1088 : 1280));
  const int per_group = one_wave ? kNormThreads / 64 : 1;
  constexpr int64_t kMostGroups = (((int64_t)1 << 32) - 1) / kNormThreads;      // a launch counts its threads in 32 bits
  const int64_t most = kMostGroups * per_group;
  for (int64_t row0 = 0; row0 < rows; row0 += most) {
    const int64_t n = rows - row0 < most ? rows - row0 : most;
    const dim3 grid((unsigned)((n + per_group - 1) / per_group)), block(kNormThreads);
    T* o = (T*)out + row0 * hidden;
    T* ro = residual_out ? (T*)residual_out + row0 * hidden : nullptr;
    const T* xr = (const T*)x + row0 * x_stride;
    const T* rr = residual ? (const T*)residual + row0 * res_stride : nullptr;
#define MVLLM_LAUNCH_N(C, W) add_rms_norm_kernel<T, C, W><<<grid, block, 0, s>>>(o, ro, xr, rr, gamma, eps, n, hidden, x_stride, res_stride)
    if (chunks <= 1) MVLLM_LAUNCH_N(1, 1);
    else if (chunks <= 2) MVLLM_LAUNCH_N(2, 1);
    else if (one_wave) MVLLM_LAUNCH_N(3, 1);
    else if (chunks <= 4) MVLLM_LAUNCH_N(1, 4);
    else if (chunks <= 8) MVLLM_LAUNCH_N(2, 4);
    else MVLLM_LAUNCH_N(4, 4);
#undef MVLLM_LAUNCH_N
    const int status = launch_status();
    if (status != MVLLM_OK) return status;
  }
  return MVLLM_OK;
}

// The norm behind a projection whose K was cut into parts (linear_small.hip): the row is the sum of the parts, plus the bias, rounded to T, and goes on as
// above, so that neither the sums nor the rounded product need a launch and a pass of their own.  A workgroup per row, a
// thread per four numbers of it, all S parts' loads under way at once: few rows wait for one memory latency, not for bandwidth.
struct PartsNorm {
  void* out;
  void* residual_out;
  const float* part;                                   // [S, gridDim.x, hidden]
  const void* bias;                                    // [hidden] or null
  const void* residual;                                // [rows, hidden] dense
  const float* gamma;
  float eps;
  int hidden;
};

template <typename T, int S, int CHUNKS, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void parts_norm_kernel(const PartsNorm a) {
  __shared__ float sums[WAVES];
  const int64_t at = (int64_t)blockIdx.x * a.hidden, size = (int64_t)gridDim.x * a.hidden;
  const T* residual = reinterpret_cast<const T*>(a.residual) + at;
  const T* bias = reinterpret_cast<const T*>(a.bias);
  float4 p[CHUNKS][S], gam[CHUNKS];
  uint2 res[CHUNKS];
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int e0 = 4 * (threadIdx.x + 64 * WAVES * c);
    if (e0 >= a.hidden) continue;
#pragma unroll
    for (int i = 0; i < S; ++i) p[c][i] = *reinterpret_cast<const float4*>(a.part + i * size + at + e0);
    res[c] = *reinterpret_cast<const uint2*>(residual + e0);
    gam[c] = *reinterpret_cast<const float4*>(a.gamma + e0);
  }
  float v[CHUNKS][4], ss = 0.f;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int e0 = 4 * (threadIdx.x + 64 * WAVES * c);
    if (e0 >= a.hidden) continue;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < S; ++i) { s[0] += p[c][i].x; s[1] += p[c][i].y; s[2] += p[c][i].z; s[3] += p[c][i].w; }
    const float r[4] = {lo_to_float<T>(res[c].x), hi_to_float<T>(res[c].x), lo_to_float<T>(res[c].y), hi_to_float<T>(res[c].y)};
    T h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (bias) s[e] += to_float(bias[e0 + e]);
      h[e] = from_float<T>(to_float(from_float<T>(s[e])) + r[e]);
      v[c][e] = to_float(h[e]);
      ss = ss + v[c][e] * v[c][e];
    }
    *reinterpret_cast<uint2*>(reinterpret_cast<T*>(a.residual_out) + at + e0) = *reinterpret_cast<const uint2*>(h);
  }
  ss = four_rows_sum(row16_sum(ss));
  if ((threadIdx.x & 63) == 0) sums[threadIdx.x >> 6] = ss;
  __syncthreads();
  ss = sums[0];
#pragma unroll
  for (int w = 1; w < WAVES; ++w) ss = ss + sums[w];
  const SharedDivisor denom(sqrtf(ss / (float)a.hidden + a.eps));
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int e0 = 4 * (threadIdx.x + 64 * WAVES * c);
    if (e0 >= a.hidden) continue;
    const T y[4] = {from_float<T>(denom.divide(v[c][0]) * gam[c].x), from_float<T>(denom.divide(v[c][1]) * gam[c].y),
                    from_float<T>(denom.divide(v[c][2]) * gam[c].z), from_float<T>(denom.divide(v[c][3]) * gam[c].w)};
    *reinterpret_cast<uint2*>(reinterpret_cast<T*>(a.out) + at + e0) = *reinterpret_cast<const uint2*>(y);
  }
}

template <typename T, int S>
static int launch_parts(const PartsNorm& a, int rows, hipStream_t stream) {
  const dim3 grid((unsigned)rows);
  if (a.hidden <= 1024) parts_norm_kernel<T, S, 1, 4><<<grid, dim3(256), 0, stream>>>(a);
  else if (a.hidden <= 2048) parts_norm_kernel<T, S, 1, 8><<<grid, dim3(512), 0, stream>>>(a);
  else if (a.hidden <= 4096) parts_norm_kernel<T, S, 1, 16><<<grid, dim3(1024), 0, stream>>>(a);
  else parts_norm_kernel<T, S, 2, 16><<<grid, dim3(1024), 0, stream>>>(a);
  return launch_status();
}

int launch_parts_norm(void* out, void* residual_out, const float* part, int splits, const void* bias, const void* residual, const float* gamma,
                      float eps, int rows, int hidden, int dtype, hipStream_t stream) {
  const PartsNorm a{out, residual_out, part, bias, residual, gamma, eps, hidden};
  const bool bf = dtype == MVLLM_BF16;
  switch (splits) {
    case 2: return bf ? launch_parts<bf16_t, 2>(a, rows, stream) : launch_parts<f16_t, 2>(a, rows, stream);
    case 3: return bf ? launch_parts<bf16_t, 3>(a, rows, stream) : launch_parts<f16_t, 3>(a, rows, stream);
    case 4: return bf ? launch_parts<bf16_t, 4>(a, rows, stream) : launch_parts<f16_t, 4>(a, rows, stream);
    default: return MVLLM_ERR_UNSUPPORTED;
  }
}

}  // namespace mvllm

using namespace mvllm;

extern "C" int mvllm_add_rms_norm(void* out, void* residual_out, const void* x, const void* residual,
                                  const float* gamma, float eps, int64_t rows, int hidden, int64_t x_row_stride,
                                  int64_t residual_row_stride, int dtype, void* stream) {
  if (dtype_size(dtype) == 0) return MVLLM_ERR_BAD_DTYPE;
  if (rows < 0 || hidden <= 0 || x_row_stride < hidden || (residual && residual_row_stride < hidden))
    return MVLLM_ERR_BAD_SHAPE;
  if (hidden % 8 != 0 || hidden > 8192) return MVLLM_ERR_UNSUPPORTED;
  if (rows == 0) return MVLLM_OK;
  if (!out || !x || !gamma) return MVLLM_ERR_NULL_POINTER;
  if (!aligned16(out) || !aligned16(x) || !aligned16(gamma) || (residual && !aligned16(residual)) ||
      (residual_out && !aligned16(residual_out)) || ((x_row_stride | residual_row_stride) & 7) != 0)
    return MVLLM_ERR_MISALIGNED;
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case MVLLM_F32:
      return launch_norm<float>(out, residual_out, x, residual, gamma, eps, rows, hidden, x_row_stride, residual_row_stride, s);
    case MVLLM_BF16:
      return launch_norm<bf16_t>(out, residual_out, x, residual, gamma, eps, rows, hidden, x_row_stride, residual_row_stride, s);
    default:
      return launch_norm<f16_t>(out, residual_out, x, residual, gamma, eps, rows, hidden, x_row_stride, residual_row_stride, s);
  }
}
