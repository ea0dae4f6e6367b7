// Gate projections of a recurrent layer: out[T, N] = act(x[T, K] W[N, K]^T + bias), N small, fp32 accumulation and fp32
// output (a recurrence's gates enter exponentials, where a 16-bit result would be a few per cent off).  Columns below
// `split` get a soft cap, cap * tanh(z / cap), the others logsigmoid of the same.
//   bf16: one workgroup = 16 or 32 rows x 16 to 80 columns; its waves take 64-wide steps of K in turn on
//         v_mfma_f32_16x16x32_bf16 and meet in LDS.
//   fp32: a 16 x 16 tile with one fp32 dot product per thread over K chunks staged in LDS.
#include "prefill_tiles.h"

#include <algorithm>

namespace mvllm {

struct GateArgs {
  float* out;              // [T, N]
  const void* x;           // [T, K]
  const void* w;           // [N, K]
  const float* bias;       // [N] or null
  int64_t x_stride;
  int rows, N, K, split;
  float cap;               // 0: no cap
};

__device__ __forceinline__ float gate_activation(const GateArgs& a, float z, int col) {
  if (a.bias) z += a.bias[col];
  if (a.cap > 0.f) z = a.cap * tanhf(z / a.cap);
  if (col >= a.split) z = fminf(z, 0.f) - log1pf(expf(-fabsf(z)));    // log sigmoid
  return z;
}

__device__ __forceinline__ uint4 load_k8(const bf16_t* row, int k, int K, bool live, bool vec) {
  uint4 r = make_uint4(0u, 0u, 0u, 0u);
  if (!live || k >= K) return r;
  if (vec && k + 8 <= K) return *reinterpret_cast<const uint4*>(row + k);
  bf16_t v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i].bits = k + i < K ? row[k + i].bits : (uint16_t)0;
  return *reinterpret_cast<const uint4*>(v);
}

constexpr int kFewRows = 512;        // up to here K is split over sixteen waves and columns over the workgroups: latency counts
// Up to here operands go straight into registers, whose call has less of a fixed part.  us so and through LDS: 8192 rows x 65, K 320 6.0 / 6.9,
// 512 7.7 / 7.0, 1024 12.3 / 8.8; 30000 x 200, K 512 61 / 65, 1024 113 / 80; 32 x 65, K 512 3.0 / 2.9, 1024 3.8 / 3.2.
constexpr int kShortK = 512;
// Up to kFewRows the line also moves with the tile's rows and columns, as repeated rows cost the address unit nothing: registers while K times (rows + columns
// of a tile) is no more.  us in registers / through LDS: 1 x 1, K 1024 2.4 / 2.9, 4096 3.6 / 4.1; 4 x 4, K 1536 3.0 / 3.2, 2048 3.4 / 3.3;
// 8 x 8, K 1024 3.0 / 3.0, 2048 4.0 / 3.4; 16 x 8, K 576 2.75 / 2.8; 16 x 16, K 704 3.2 / 2.9; 4 x 2, K 2048 3.2 / 3.3, 3072 3.8 / 3.7, 4096 4.3 / 4.1.
constexpr int64_t kRegisterLines = 16384;
constexpr int kManyRows = 4096;      // from here 32 rows to a workgroup: they fill the CUs and read W half as often

// Whole rows of x and W through LDS: a matrix operand's lanes are sixteen different rows, which a CU's address unit takes at 16 B per
// clock; eight lanes to a 128-byte line it takes at 64, and that is what bounds the call (W is read again by every workgroup).  A wave has its own
// 64 values of K per step and its own ring of S panels of 16 (RT + NT) rows of them, so it waits for nobody until the sums
// meet: chunk c of K belongs to partial sum c % (SK kSums), in wave c % SK.  A row's eight pieces trade places by the row's
// number, which spreads the banks.  Rows and columns past the end repeat the last one and are not stored; copies past a wave's
// last step run with an empty descriptor.
// Sums are those of gate_linear_bf16_kernel to the bit.  us with operands straight into registers and so: 32 rows x 65, K 4096 8.9 / 4.4; 512 x 65, K 2048
// 5.6 / 3.7; 2048 x 65, K 4096 22.6 / 10.7; 8192 x 65, K 2048 21.6 / 11.8 (3.0 TB/s of x; 6.8 at the copy's rate); 20000 x 65 50 / 31.
template <int RT, int NT, int SK, int kSums, int S>
__global__ __launch_bounds__(64 * SK) void gate_linear_ring_kernel(const GateArgs a) {
  constexpr int kPanel = 2 * (RT + NT) * 1024, kCopies = 2 * (RT + NT), kParts = SK * kSums;
  static_assert(S >= 2 && kCopies * (S - 2) <= 63 && S * SK * kPanel <= 160 * 1024 && kParts * RT * NT * 1024 <= S * SK * kPanel, "waits, LDS");
  __shared__ __attribute__((aligned(1024))) char lds[S * SK * kPanel];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row0 = blockIdx.x * 16 * RT, col0 = blockIdx.y * 16 * NT;
  const int rows = min(a.rows - row0, 16 * RT), cols = min(a.N - col0, 16 * NT);
  const uint32_t x_row = (uint32_t)a.x_stride * 2u, w_row = (uint32_t)a.K * 2u;
  const char* x = reinterpret_cast<const char*>(a.x) + (int64_t)row0 * a.x_stride * 2;
  const char* w = reinterpret_cast<const char*>(a.w) + (int64_t)col0 * a.K * 2;
  const int r8 = lane >> 3;
  const uint32_t piece = (uint32_t)(((lane & 7) ^ r8) << 4);
  uint32_t from[kCopies];
  static_for<kCopies>([&](auto I) {
    constexpr int i = decltype(I)::value;
    if constexpr (i < 2 * RT) from[i] = (uint32_t)min(8 * i + r8, rows - 1) * x_row + piece;
    else from[i] = (uint32_t)min(8 * (i - 2 * RT) + r8, cols - 1) * w_row + piece;
  });
  const int chunks = a.K / 64, steps = (chunks - wave + SK - 1) / SK;
  const uint32_t x_bytes = (uint32_t)(rows - 1) * x_row + w_row, w_bytes = (uint32_t)cols * w_row;
  const uint32_t lds0 = lds_address(lds) + wave * (S * kPanel);
  auto copy = [&](int step, int buffer) __attribute__((always_inline)) {
    const bool live = step < steps;
    const v4i x_rows = make_rsrc(x, live ? x_bytes : 0u), w_rows = make_rsrc(w, live ? w_bytes : 0u);
    const uint32_t at = live ? (uint32_t)(step * SK + wave) * 128u : 0u, base = lds0 + buffer * kPanel;
    static_for<kCopies>([&](auto I) {
      constexpr int i = decltype(I)::value;
      dma16_to_lds_at<i * 1024>(i < 2 * RT ? x_rows : w_rows, from[i], at, base);
    });
  };
  v4f acc[kSums][RT][NT];
#pragma unroll
  for (int c = 0; c < kSums; ++c)
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[c][r][n] = v4f{0.f, 0.f, 0.f, 0.f};
  static_for<S - 1>([&](auto I) { copy(decltype(I)::value, decltype(I)::value); });
  // row l % 16 of a tile (row l % 8 of one of its two blocks), the 32 bytes l / 16 of the 128: piece 2 (l / 16) + half
  const char* frag = lds + wave * (S * kPanel) + ((lane >> 3) & 1) * 1024 + (lane & 7) * 128;
  const int p0 = ((2 * (lane >> 4)) ^ (lane & 7)) << 4, p1 = p0 ^ 16;
  int buffer = 0;
  for (int first = 0; first < steps; first += kSums)
    static_for<kSums>([&](auto C) {
      constexpr int c = decltype(C)::value;
      if (first + c >= steps) return;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the panel read before takes the next copies
      dma_wait_but<kCopies * (S - 2)>();
      copy(first + c + S - 1, buffer == 0 ? S - 1 : buffer - 1);
      const char* st = frag + buffer * kPanel;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int p = half ? p1 : p0;
        uint4 xf[RT], wf[NT];
#pragma unroll
        for (int r = 0; r < RT; ++r) xf[r] = *reinterpret_cast<const uint4*>(st + 2048 * r + p);
#pragma unroll
        for (int n = 0; n < NT; ++n) wf[n] = *reinterpret_cast<const uint4*>(st + 2048 * (RT + n) + p);
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int n = 0; n < NT; ++n) acc[c][r][n] = mfma16x16x32<bf16_t>(wf[n], xf[r], acc[c][r][n]);
      }
      buffer = buffer + 1 == S ? 0 : buffer + 1;
    });
  // lane holds row l % 16, columns 4 (l / 16) + r of every tile; the activations are spread over the workgroup
  dma_wait_all();
  workgroup_barrier();                                     // the rings are read and written to their end
  float* part = reinterpret_cast<float*>(lds);             // [kParts][RT][NT][64 lanes][4]
#pragma unroll
  for (int c = 0; c < kSums; ++c)
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int n = 0; n < NT; ++n)
        *reinterpret_cast<float4*>(part + ((((c * SK + wave) * RT + r) * NT + n) * 64 + lane) * 4) =
            make_float4(acc[c][r][n][0], acc[c][r][n][1], acc[c][r][n][2], acc[c][r][n][3]);
  __syncthreads();
  for (int t = threadIdx.x; t < 256 * RT * NT; t += 64 * SK) {
    const int tile = t >> 8, c = (t >> 4) & 15, row = 16 * (tile / NT) + (t & 15), col = 16 * (tile % NT) + c;
    if (row >= rows || col >= cols) continue;
    float z = 0.f;
#pragma unroll
    for (int i = 0; i < kParts; ++i) z += part[((i * RT * NT + tile) * 64 + 16 * (c >> 2) + (t & 15)) * 4 + (c & 3)];
    a.out[(int64_t)(row0 + row) * a.N + col0 + col] = gate_activation(a, z, col0 + col);
  }
}

// Short or odd K: operands straight into registers.  kWaves waves share K; NT column tiles per workgroup (one pass over x for all of them); kFull: K is a multiple of 64 and rows are 16-byte
// aligned, so that loads need no guards (rows and columns past the end load the last one and are not stored).
template <int kWaves, int NT, bool kFull>
__global__ __launch_bounds__(64 * kWaves) void gate_linear_bf16_kernel(const GateArgs a, bool vec) {
  __shared__ float4 part[kWaves][NT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = blockIdx.x * 16 + (lane & 15), col0 = blockIdx.y * 16 * NT + (lane & 15);
  const int k0 = 8 * (lane >> 4);
  const bf16_t* x = reinterpret_cast<const bf16_t*>(a.x) + (int64_t)(kFull ? min(row, a.rows - 1) : row) * a.x_stride;
  const bf16_t* w[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int col = col0 + 16 * n;
    w[n] = reinterpret_cast<const bf16_t*>(a.w) + (int64_t)(kFull ? min(col, a.N - 1) : col) * a.K;
  }
  v4f acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = v4f{0.f, 0.f, 0.f, 0.f};
  if constexpr (kFull) {
#pragma unroll 4
    for (int k = 64 * wave + 2 * k0; k < a.K; k += 64 * kWaves) {      // a lane's 32 bytes: whole lines per row and wave
#pragma unroll
      for (int half = 0; half < 16; half += 8) {
        const uint4 xv = *reinterpret_cast<const uint4*>(x + k + half);
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = mfma16x16x32<bf16_t>(*reinterpret_cast<const uint4*>(w[n] + k + half), xv, acc[n]);
      }
    }
  } else {
#pragma unroll 4
    for (int k = 32 * wave; k < a.K; k += 32 * kWaves) {
      const uint4 xv = load_k8(x, k + k0, a.K, row < a.rows, vec);
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[n] = mfma16x16x32<bf16_t>(load_k8(w[n], k + k0, a.K, col0 + 16 * n < a.N, vec), xv, acc[n]);
    }
  }
  // lane holds row l % 16, columns 4 (l / 16) + r of every tile; the activations are spread over the workgroup
#pragma unroll
  for (int n = 0; n < NT; ++n) part[wave][n][lane] = make_float4(acc[n][0], acc[n][1], acc[n][2], acc[n][3]);
  __syncthreads();
  for (int t = threadIdx.x; t < 256 * NT; t += 64 * kWaves) {
    const int n = t >> 8, c = (t >> 4) & 15, out_row = blockIdx.x * 16 + (t & 15), out_col = (blockIdx.y * NT + n) * 16 + c;
    if (out_row >= a.rows || out_col >= a.N) continue;
    float z = 0.f;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) z += reinterpret_cast<const float*>(&part[i][n][16 * (c >> 2) + (t & 15)])[c & 3];
    a.out[(int64_t)out_row * a.N + out_col] = gate_activation(a, z, out_col);
  }
}

__global__ __launch_bounds__(256) void gate_linear_f32_kernel(const GateArgs a) {
  constexpr int kStep = 64;
  __shared__ float xs[16][kStep + 1], ws[16][kStep + 1];
  const int r = threadIdx.x >> 4, c = threadIdx.x & 15;
  const int row = blockIdx.x * 16 + r, col = blockIdx.y * 16 + c;
  const float* x = reinterpret_cast<const float*>(a.x);
  const float* w = reinterpret_cast<const float*>(a.w);
  float acc = 0.f;
  for (int k0 = 0; k0 < a.K; k0 += kStep) {
    for (int i = threadIdx.x; i < 16 * kStep; i += 256) {
      const int rr = i / kStep, k = i % kStep;
      const int xr = blockIdx.x * 16 + rr, wr = blockIdx.y * 16 + rr;
      xs[rr][k] = xr < a.rows && k0 + k < a.K ? x[(int64_t)xr * a.x_stride + k0 + k] : 0.f;
      ws[rr][k] = wr < a.N && k0 + k < a.K ? w[(int64_t)wr * a.K + k0 + k] : 0.f;
    }
    __syncthreads();
#pragma unroll 16
    for (int k = 0; k < kStep; ++k) acc = fmaf(xs[r][k], ws[c][k], acc);
    __syncthreads();
  }
  if (row < a.rows && col < a.N) a.out[(int64_t)row * a.N + col] = gate_activation(a, acc, col);
}

template <int NT>
static void launch_many(const GateArgs& a, bool ring, hipStream_t s) {
  constexpr auto stages = [](int rt) { const int n = 160 / (8 * (rt + NT)); return n < 4 ? n : 4; };
  const unsigned y = (unsigned)((a.N + 16 * NT - 1) / (16 * NT));
  const dim3 grid16((unsigned)((a.rows + 15) / 16), y), grid32((unsigned)((a.rows + 31) / 32), y);
  if (!ring) gate_linear_bf16_kernel<8, NT, true><<<grid16, dim3(512), 0, s>>>(a, true);
  else if (a.rows > kManyRows) gate_linear_ring_kernel<2, NT, 4, 2, stages(2)><<<grid32, dim3(256), 0, s>>>(a);
  else gate_linear_ring_kernel<1, NT, 4, 2, stages(1)><<<grid16, dim3(256), 0, s>>>(a);
}

}  // namespace mvllm

using namespace mvllm;

extern "C" int mvllm_gate_linear(float* out, const void* x, int64_t x_row_stride, const void* w, const float* bias,
                                 int64_t rows, int N, int K, int split, float cap, int dtype, void* stream) {
  if (dtype_size(dtype) == 0) return MVLLM_ERR_BAD_DTYPE;
  if (rows < 0 || N <= 0 || K <= 0 || split < 0 || split > N || x_row_stride < K || !(cap >= 0.f)) return MVLLM_ERR_BAD_SHAPE;
  if (dtype == MVLLM_F16 || rows > (1 << 30) || N > 65535 * 16) return MVLLM_ERR_UNSUPPORTED;
  if (rows == 0) return MVLLM_OK;
  if (!out || !x || !w) return MVLLM_ERR_NULL_POINTER;
  GateArgs a;
  a.out = out; a.x = x; a.w = w; a.bias = bias; a.x_stride = x_row_stride; a.rows = (int)rows; a.N = N; a.K = K;
  a.split = split; a.cap = cap;
  const unsigned tiles = (unsigned)((rows + 15) / 16), columns = (unsigned)((N + 15) / 16);
  hipStream_t s = (hipStream_t)stream;
  const bool vec = K % 8 == 0 && x_row_stride % 8 == 0 && aligned16(x) && aligned16(w), full = vec && K % 64 == 0;
  const bool wide = rows > kFewRows || (int64_t)K * (std::min((int)rows, 16) + std::min(N, 16)) > kRegisterLines;
  const bool ring = full && wide && K > kShortK && std::max(32 * x_row_stride, 80 * (int64_t)K) * 2 < (int64_t)1 << 32;   // a descriptor's offsets
  if (dtype == MVLLM_F32) gate_linear_f32_kernel<<<dim3(tiles, columns), dim3(256), 0, s>>>(a);
  else if (!full) gate_linear_bf16_kernel<4, 1, false><<<dim3(tiles, columns), dim3(256), 0, s>>>(a, vec);
  else if (rows <= kFewRows && ring) gate_linear_ring_kernel<1, 1, 16, 1, 2><<<dim3(tiles, columns), dim3(1024), 0, s>>>(a);
  else if (rows <= kFewRows) gate_linear_bf16_kernel<16, 1, true><<<dim3(tiles, columns), dim3(1024), 0, s>>>(a, vec);
  else if (columns == 1) launch_many<1>(a, ring, s);
  else if (columns == 2) launch_many<2>(a, ring, s);
  else if (columns == 3) launch_many<3>(a, ring, s);
  else if (columns == 4) launch_many<4>(a, ring, s);
  else launch_many<5>(a, ring, s);
  return launch_status();
}
