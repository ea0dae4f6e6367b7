// Linear layer for the few rows of a decode step: out[M, N] = x[M, K] W[N, K]^T + bias, M <= 64, bf16 / fp16.
// The caller's projections around the attention path (src/myvllm/models/qwen3.py:90-94, 118 and the MLP, :121-160;
// layers/linear.py) are library GEMMs in the reference.  Such a product reads a few MB to a few hundred MB of weights
// once, from HBM: what bounds it is that stream, and beside it the address unit of a CU, which takes a 16-byte load of a
// wave at 64 B per clock where four neighbouring lanes share 64 bytes and at 16 B where they do not (a matrix
// operand's lanes are sixteen different rows).  Hence two kernels:
//   linear_rows_kernel (very few rows): weights and x straight into registers, eight rows x 128 bytes per load.
//   linear_ring_kernel (more rows): W and x through a ring of tiles in LDS, copied as whole 128-byte lines.
// Both read a weight once, but for few columns' ring, whose tiles of 16 rows are apart (rows_apart).  A sum's order depends on (M, N, K) and, from kStreamBytes of weights on, on the column; a long K with few columns is cut into
// parts where the caller brings room for their sums (linear_split).
// mvllm_norm_linear_small_m is the same product with the launches around it folded in: the residual add + RMSNorm in
// front of the layer's first projections (src/myvllm/models/qwen3.py:197-212 through layers/layernorm.py:9-28) as
// the kernel's prologue (linear_norm_kernel), and SiluAndMul behind the gate/up projection (layers/activation.py:15-18) as
// its epilogue, each rounding where the separate launch rounds.  mvllm_linear_add_rms_norm is the product in parts of K with that norm behind it.
#include "prefill_tiles.h"

#pragma clang fp contract(off)

namespace mvllm {

struct LinearSplit { int columns, splits; };               // of K; splits 1: whole, with ring_columns

struct LinearArgs {
  void* out;
  const void* x;
  const void* w;
  const void* bias;       // [N] in the element type, or null
  int64_t x_row_stride;   // elements between rows of x
  int M, N, K;
  // norm: x is first replaced by rms_norm(x + residual) * gamma, as mvllm_add_rms_norm computes it
  const void* residual;   // [M, K] contiguous, or null (then the norm of x alone)
  void* residual_out;     // [M, K] contiguous: x + residual in the element type; must not alias x or residual
  const float* gamma;     // [K]
  float eps;
  int row_tiles;          // norm: tiles of 16 rows, a workgroup per column tile each
  int gelu;               // plain product only: the result through the tanh form of gelu
  int part_steps;         // steps of the ring in a part of K
  float* part;            // plain product only: partial sums [gridDim.y, M, N] of the splits of K, or null
  LinearSplit split;      // with part
  bool leave_parts;       // the next launch adds the parts up
};

// silu(g) * u with the roundings of the two tensor operations (activation.hip): silu in fp32 rounded to T, then the
// product rounded to T
template <typename T>
__device__ __forceinline__ T silu_mul_rounded(T g, T u) {
  const float a = to_float(g);
  const float s = to_float(from_float<T>(a / (1.0f + __expf(-a))));
  return from_float<T>(s * to_float(u));
}

template <typename T>
__device__ __forceinline__ void unpack8(uint4 w, float (&x)[8]) {
  x[0] = lo_to_float<T>(w.x); x[1] = hi_to_float<T>(w.x);
  x[2] = lo_to_float<T>(w.y); x[3] = hi_to_float<T>(w.y);
  x[4] = lo_to_float<T>(w.z); x[5] = hi_to_float<T>(w.z);
  x[6] = lo_to_float<T>(w.w); x[7] = hi_to_float<T>(w.w);
}
template <typename T>
__device__ __forceinline__ uint4 pack8(const float (&x)[8]) {
  return make_uint4(pack2<T>(x[0], x[1]), pack2<T>(x[2], x[3]), pack2<T>(x[4], x[5]), pack2<T>(x[6], x[7]));
}

// What follows a product: bias, gelu or the gated unit, rounding.  `s`: out[m][j .. j + 3]; GLU: `u` the up columns that meet them.
template <typename T, bool GLU>
__device__ __forceinline__ void finish_four(const LinearArgs& a, int m, int j, float (&s)[4], float (&u)[4]) {
  const int out_cols = GLU ? a.N / 2 : a.N;
  if (m >= a.M || j >= out_cols) return;
  if (a.bias) {
    const T* bp = reinterpret_cast<const T*>(a.bias) + j;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s[r] += to_float(bp[r]);
      if (GLU) u[r] += to_float(bp[out_cols + r]);
    }
  }
  T r4[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if constexpr (GLU) r4[r] = silu_mul_rounded<T>(from_float<T>(s[r]), from_float<T>(u[r]));
    else r4[r] = from_float<T>(a.gelu ? gelu_tanh(s[r]) : s[r]);
  }
  *reinterpret_cast<uint2*>(reinterpret_cast<T*>(a.out) + (int64_t)m * out_cols + j) = *reinterpret_cast<const uint2*>(r4);
}

// Very few rows.  A load of a wave covers 8 rows x 64 values of K, whole 128-byte lines: lane l holds 8 values of row
// l % 8 from piece 4 (l / 8 % 2) + l / 16 on.  As operands of v_mfma_f32_16x16x32 such registers are 16 "rows" (row, half of the 64
// values), so that a product of a weight and an x register is valid where the halves agree, half of the results: the matrix
// unit, idle otherwise, does twice the work, and the halves meet in the sum over the waves.  (Sixteen rows x 64 bytes per
// load, the operand's own layout: 26.7 against 20.1 us at N 4096, K 12288 with all else equal; the kernel as a whole against the one it
// replaces, one row, us: 18.8 / 30.2 there, 33.7 / 40.0 at 24576 x 4096 (6.0 TB/s), 10.9 / 16.1 at 6144 x 4096, 3.5 / 4.4 at 1024 x 2048.)
// Waves split K; each walks its share in chunks of U loads per weight tile, the next chunk on its way while this one is multiplied.
// WT tiles of 8 weight rows per workgroup; GLU: the first half of them gate columns, the second half the up columns that meet them.
template <typename T, int WT, int U, int W, bool GLU>
__global__ __launch_bounds__(64 * W) void linear_rows_kernel(const LinearArgs a) {
  static_assert(!GLU || WT % 2 == 0, "gate and up tiles come in pairs");
  __shared__ float4 part[W * WT * 64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row8 = lane & 7, piece = ((lane >> 3) & 1) * 4 + (lane >> 4);
  const int ksl = a.K / W;
  const int koff = wave * ksl + piece * 8;
  const int out_cols = GLU ? a.N / 2 : a.N;
  const int j0 = blockIdx.x * (GLU ? WT * 4 : WT * 8);     // first output column
  const T* wp[WT];
#pragma unroll
  for (int wt = 0; wt < WT; ++wt) {
    const int t = GLU ? wt % (WT / 2) : wt;
    const int row = min(j0 + 8 * t + row8, out_cols - 1) + (GLU && wt >= WT / 2 ? out_cols : 0);     // rows past the last repeat it
    wp[wt] = reinterpret_cast<const T*>(a.w) + (int64_t)row * a.K + koff;
  }
  const T* xp = reinterpret_cast<const T*>(a.x) + (int64_t)min(row8, a.M - 1) * a.x_row_stride + koff;
  v4f acc[WT];
#pragma unroll
  for (int wt = 0; wt < WT; ++wt) acc[wt] = (v4f){0.f, 0.f, 0.f, 0.f};
  struct Chunk { uint4 w[WT][U], x[U]; };
  Chunk even, odd;
  auto load = [&](Chunk& c, int k) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int wt = 0; wt < WT; ++wt) c.w[wt][u] = load16_stream(wp[wt] + k + 64 * u);
#pragma unroll
    for (int u = 0; u < U; ++u) c.x[u] = *reinterpret_cast<const uint4*>(xp + k + 64 * u);
  };
  auto multiply = [&](const Chunk& c) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int wt = 0; wt < WT; ++wt) acc[wt] = mfma16x16x32<T>(c.w[wt][u], c.x[u], acc[wt]);
  };
  constexpr int kStep = 64 * U;
  int k = 0;
  load(even, 0);
  for (; k + 2 * kStep < ksl; k += 2 * kStep) {            // loads stay in front of the products of the chunk before
    load(odd, k + kStep);
    __builtin_amdgcn_sched_barrier(0);
    multiply(even);
    __builtin_amdgcn_sched_barrier(0);
    load(even, k + 2 * kStep);
    __builtin_amdgcn_sched_barrier(0);
    multiply(odd);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (k + kStep < ksl) {
    load(odd, k + kStep);
    multiply(even);
    multiply(odd);
  } else {
    multiply(even);
  }
#pragma unroll
  for (int wt = 0; wt < WT; ++wt) part[(wave * WT + wt) * 64 + lane] = make_float4(acc[wt][0], acc[wt][1], acc[wt][2], acc[wt][3]);
  __syncthreads();
  // 16 threads a tile: row m, columns 4 quad .. + 3; the first half's result is in lane 16 quad + m, the second's in 16 (quad + 2) + 8 + m.  GLU: as many
  // again for the up tiles, half a wave on: the waves' sums one after the other are what few columns wait for (us at one row, gate and up
  // by one thread / by two: 512 x 512 3.08 / 2.89, 1024 x 1536 4.12 / 3.93, 2048 x 1024 3.65 / 3.52, 11456 x 1024 6.81 / 6.63)
  constexpr int kOutTiles = GLU ? WT / 2 : WT, kLanes = kOutTiles * 16;
  static_assert(!GLU || kLanes <= 32, "gate and up threads meet within a wave");
  const int t = GLU ? threadIdx.x & 31 : threadIdx.x;
  if (threadIdx.x < (GLU ? 64 : kLanes) && t < kLanes) {
    const int quad = t & 1, wt = (t >> 1) % kOutTiles, m = (t >> 1) / kOutTiles;
    const float4* of = part + (GLU && threadIdx.x >= 32 ? wt + WT / 2 : wt) * 64 + 16 * quad + m;
    float s[4] = {0.f, 0.f, 0.f, 0.f}, u[4];
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float4 lo = of[w * WT * 64], hi = of[w * WT * 64 + 40];
      s[0] += lo.x + hi.x; s[1] += lo.y + hi.y; s[2] += lo.z + hi.z; s[3] += lo.w + hi.w;
    }
    if constexpr (GLU) {
#pragma unroll
      for (int r = 0; r < 4; ++r) u[r] = __shfl_down(s[r], 32, 64);
      if (threadIdx.x >= 32) return;
    }
    finish_four<T, GLU>(a, m, j0 + 8 * wt + 4 * quad, s, u);
  }
}

// More rows: a workgroup owns 16 CT SC output columns and MT * 16 rows, all or (blockIdx.z) some of them.  SK waves split the 64 SK values of a stage
// between them, SC such groups the columns; a stage is WB + XB blocks of 8 rows x 128 bytes per 64 values, copied into a ring of
// S of them (buffer loads to LDS: eight lines a wave and copy, no registers, S - 1 stages under way; a row's eight pieces
// trade places by the row's number, which spreads both the copies' and the reads' banks).  One barrier a stage: behind it
// this stage's copies are there and the stage before has been read by all, so its place takes the next copies.  Past the last stage
// copies go on with an empty descriptor, which keeps the count that a wave waits for.
// us against the form before it (a workgroup per 16 columns and 16 rows, operands straight into registers), 16 / 32 / 64 rows: 4096 x 1024 4.0 / 4.7 / 5.6
// against 4.7 / 6.4 / 9.7, 4096 x 12288 21.5 / 28.1 / 36.4 against 34.8 / 50 / 90 (16.8 at 6 TB/s), 24576 x 4096 with GLU 35.7 / 39.4 / 46.6 (4.3 TB/s)
// against 58 / 95 / 178.
// GLU: gate and up rows in turns of eight, so that a tile's lanes hold gates (l / 16 < 2) and, 32 lanes on, what meets them.
// NT: the weights' lines are marked as read once, +5 to 10 % where the call's weights are a stream from HBM; small
// weights of a small model may still be in the memory-side cache from the step before (4.4 against 5.8 us at 1024 x 3072, 16 rows).
template <typename T, int MT, int CT, int SK, int SC, int S, bool NT, bool GLU>
__global__ __launch_bounds__(64 * SK * SC) void linear_ring_kernel(const LinearArgs a) {
  constexpr int NW = SK * SC, WB = 2 * CT * SC, XB = 2 * MT;
  constexpr int kPanel = (WB + XB) * 1024, kStage = SK * kPanel, kCopies = (WB + XB) / SC;
  static_assert((WB + XB) % SC == 0 && S >= 2 && kCopies * (S - 2) <= 63 && S * kStage <= 160 * 1024, "copies of a wave, waits, LDS");
  static_assert(NW * MT * CT * 1024 <= S * kStage, "the sums reuse the ring");
  __shared__ __attribute__((aligned(1024))) char lds[S * kStage];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sk = wave % SK, sc = wave / SK;
  const int out_cols = GLU ? a.N / 2 : a.N;
  constexpr int kSpan = (GLU ? 8 : 16) * CT * SC;          // output columns of the workgroup
  const int first = blockIdx.x * kSpan, left = out_cols - first;
  const uint32_t row_bytes = (uint32_t)a.K * 2u;
  const char* w0 = reinterpret_cast<const char*>(a.w) + (int64_t)first * row_bytes;
  const uint32_t w_bytes = (uint32_t)min(left, kSpan) * row_bytes;
  const int m0 = 16 * MT * (int)blockIdx.z, rows = min(a.M - m0, 16 * MT);
  const char* x0 = reinterpret_cast<const char*>(a.x) + (int64_t)m0 * a.x_row_stride * 2;
  const uint32_t x_bytes = ((uint32_t)(rows - 1) * (uint32_t)a.x_row_stride + (uint32_t)a.K) * 2u;
  const int r8 = lane >> 3;
  const uint32_t piece = (uint32_t)(sk * 128 + (((lane & 7) ^ r8) << 4));
  uint32_t from[kCopies];                                  // rows past the last repeat it
  static_for<kCopies>([&](auto I) {
    constexpr int i = decltype(I)::value;
    const int b = i * SC + sc;
    if constexpr (i < 2 * CT) from[i] = (uint32_t)min(8 * (GLU ? b >> 1 : b) + r8, left - 1) * row_bytes + piece;
    else from[i] = (uint32_t)min(8 * (b - WB) + r8, rows - 1) * (uint32_t)a.x_row_stride * 2u + piece;
  });
  const int step0 = a.part_steps * (int)blockIdx.y, steps = min(a.K / (64 * SK) - step0, a.part_steps);    // of this workgroup's part of K
  // Rows a multiple of 4 KB long start in the same channel of the L2 and of the memory: workgroups that walk K in step would all read
  // from a few of them, so neighbours on an XCD start a quarter of the steps apart.  us at 16 / 33 / 64 rows without and with: 24576 x 4096 with GLU 34.2 /
  // 41.8 / 45.9 and 32.3 / 41.0 / 39.0, 6144 x 4096 14.3 / 14.9 / 17.2 and 12.4 / 13.5 / 16.6, 12288 x 2048 with GLU 13.1 / 13.8 / 15.5 and 12.5 / 13.0 / 14.7.
  const int turn = NT && a.K % 2048 == 0 ? (int)(blockIdx.x >> 3 & 3) * (steps >> 2) : 0;
  const uint32_t lds0 = lds_address(lds) + sk * kPanel + sc * 1024;
  auto copy = [&](int step, int buffer) __attribute__((always_inline)) {
    const bool live = step < steps;
    const v4i x_rows = make_rsrc(x0, live ? x_bytes : 0u);
    const v4i w_rows = make_rsrc(w0, live ? w_bytes : 0u);
    const v4i up_rows = GLU ? make_rsrc(w0 + (int64_t)out_cols * row_bytes, live ? w_bytes : 0u) : w_rows;
    const uint32_t at = live ? (uint32_t)(step0 + (step < steps - turn ? step + turn : step + turn - steps)) * (SK * 128) : 0u, base = lds0 + buffer * kStage;
    static_for<kCopies>([&](auto I) {
      constexpr int i = decltype(I)::value;
      if constexpr (i < 2 * CT) dma16_to_lds_at<i * SC * 1024, NT>(GLU && ((i * SC + sc) & 1) ? up_rows : w_rows, from[i], at, base);
      else dma16_to_lds_at<i * SC * 1024>(x_rows, from[i], at, base);
    });
  };
  v4f acc[MT][CT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) acc[mt][ct] = (v4f){0.f, 0.f, 0.f, 0.f};
  static_for<S - 1>([&](auto I) { copy(decltype(I)::value, decltype(I)::value); });
  // fragments of v_mfma_f32_16x16x32: row l % 16 of a tile (row l % 8 of one of its two blocks), piece 4 kk + l / 16
  const char* frag = lds + sk * kPanel + ((lane >> 3) & 1) * 1024 + (lane & 7) * 128;
  const int p0 = ((lane >> 4) ^ (lane & 7)) << 4, p1 = p0 ^ 64;
  int buffer = 0;
  for (int step = 0; step < steps; ++step) {
    dma_wait_but<kCopies * (S - 2)>();
    workgroup_barrier();
    copy(step + S - 1, buffer == 0 ? S - 1 : buffer - 1);
    const char* st = frag + buffer * kStage;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int p = kk ? p1 : p0;
      uint4 wf[CT], xf[MT];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) wf[ct] = *reinterpret_cast<const uint4*>(st + (sc * CT + ct) * 2048 + p);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) xf[mt] = *reinterpret_cast<const uint4*>(st + (WB + 2 * mt) * 1024 + p);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt][ct] = mfma16x16x32<T>(wf[ct], xf[mt], acc[mt][ct]);
    }
    buffer = buffer + 1 == S ? 0 : buffer + 1;
  }
  // lane l of a tile holds out[16 mt + l % 16][weight rows 4 (l / 16) .. + 3 of the tile]
  const int col = lane & 15, cls = lane >> 4;
  dma_wait_all();
  workgroup_barrier();                                     // the ring is read and written to its end
  float4* part = reinterpret_cast<float4*>(lds);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
      part[((wave * MT + mt) * CT + ct) * 64 + lane] = make_float4(acc[mt][ct][0], acc[mt][ct][1], acc[mt][ct][2], acc[mt][ct][3]);
  __syncthreads();
  for (int t = wave; t < SC * MT * CT; t += NW) {
    const int c = t / (MT * CT), mc = t % (MT * CT);
    float s[4] = {0.f, 0.f, 0.f, 0.f}, u[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < SK; ++k) {
      const float4 p = part[((c * SK + k) * MT * CT + mc) * 64 + lane];
      s[0] += p.x; s[1] += p.y; s[2] += p.z; s[3] += p.w;
    }
    if constexpr (GLU) {
#pragma unroll
      for (int r = 0; r < 4; ++r) u[r] = __shfl_xor(s[r], 32, 64);
      if (cls >= 2) continue;
    }
    const int m = m0 + 16 * (mc / CT) + col, j = first + (GLU ? 8 : 16) * (c * CT + mc % CT) + 4 * cls;
    if (!GLU && a.part) {
      if (m < a.M && j < a.N) *reinterpret_cast<float4*>(a.part + ((int64_t)blockIdx.y * a.M + m) * a.N + j) = make_float4(s[0], s[1], s[2], s[3]);
    } else {
      finish_four<T, GLU>(a, m, j, s, u);
    }
  }
}

// The sums of the splits of K, four outputs a thread.
template <typename T>
__global__ __launch_bounds__(256) void linear_sum_kernel(const LinearArgs a, int splits) {
  const int64_t at = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x), size = (int64_t)a.M * a.N;
  if (at >= size) return;
  float s[4] = {0.f, 0.f, 0.f, 0.f}, u[4];
#pragma unroll 4
  for (int i = 0; i < splits; ++i) {
    const float4 p = *reinterpret_cast<const float4*>(a.part + i * size + at);
    s[0] += p.x; s[1] += p.y; s[2] += p.z; s[3] += p.w;
  }
  const int m = (int)(at / a.N);
  finish_four<T, false>(a, m, (int)(at - (int64_t)m * a.N), s, u);
}

// The product behind the residual add and norm: K = 512 P, eight waves, each with 64 P values of K, 16 rows of x and 16 CT weight rows per
// workgroup.  Every workgroup needs every row, so each of them forms h = x + residual for its rows, a wave per row, and leaves the rounded
// h / sqrt(mean h^2 + eps) * gamma in LDS as the second operand: the value the separate norm launch would have written, without
// the launch.  Workgroup b < M also writes row b of h (the next residual).  The wave's weights are asked for behind the rows and are on their
// way meanwhile; they go through a place in LDS of the wave's own, because whole lines are loaded (see the top of this file).
// us at 1 / 16 rows, before (operands straight into registers, rows normalised once per 16 lanes that share them) and now:
// 4096 x 1024 6.2 / 7.4 and 4.0 / 5.5 (the product alone 3.8 / 4.0), 6144 x 1024 with GLU 8.4 / 10.7 and 5.1 / 6.6, 4096 x 2048 9.3 /
// 11.3 and 5.8 / 8.7.
template <typename T, int CT, int P, bool GLU>
__global__ __launch_bounds__(512) void linear_norm_kernel(const LinearArgs a) {
  constexpr int W = 8, kPanel = 2048;                      // waves; bytes of 16 rows x 64 values: two blocks of 8 rows, as in linear_ring_kernel
  constexpr int kX = W * P * kPanel, kW = W * CT * kPanel;
  __shared__ __attribute__((aligned(1024))) char lds[kX + kW];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = 16 * blockIdx.y, mrows = min(a.M - m0, 16);
  const int out_cols = GLU ? a.N / 2 : a.N, K = 512 * P;
  const int first = blockIdx.x * (GLU ? 8 : 16) * CT, left = out_cols - first;
  // ---- loads: rows wave and wave + 8 (8 values of K per lane and chunk of 512), gamma, then the weights of 64 P values ----
  uint4 x[2][P], res[2][P];
  float4 gam[P][2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = wave + 8 * i;
    if (row < mrows) {
      const T* xp = reinterpret_cast<const T*>(a.x) + (int64_t)(m0 + row) * a.x_row_stride + 8 * lane;
      const T* rp = reinterpret_cast<const T*>(a.residual) + (int64_t)(m0 + row) * K + 8 * lane;
#pragma unroll
      for (int c = 0; c < P; ++c) {
        x[i][c] = *reinterpret_cast<const uint4*>(xp + 512 * c);
        if (a.residual) res[i][c] = *reinterpret_cast<const uint4*>(rp + 512 * c);
      }
    }
  }
#pragma unroll
  for (int c = 0; c < P; ++c) {
    gam[c][0] = *reinterpret_cast<const float4*>(a.gamma + 512 * c + 8 * lane);
    gam[c][1] = *reinterpret_cast<const float4*>(a.gamma + 512 * c + 8 * lane + 4);
  }
  const int r8 = lane >> 3;
  uint4 w[P][CT][2];
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int b = 0; b < 2; ++b) {                        // GLU: block 0 of a tile gate rows, block 1 up rows; rows past the last repeat it
        const int row = GLU ? min(8 * ct + r8, left - 1) + first + (b ? out_cols : 0) : first + min(16 * ct + 8 * b + r8, left - 1);
        const T* wp = reinterpret_cast<const T*>(a.w) + (int64_t)row * K + 64 * (wave * P + p) + 8 * (lane & 7);
        w[p][ct][b] = a.row_tiles > 1 ? *reinterpret_cast<const uint4*>(wp) : load16_stream(wp);
      }
  // ---- rows: sum, norm, into LDS: panel k / 64, block row / 8, row row % 8, piece k / 8 % 8 with its place changed by the row ----
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = wave + 8 * i;
    if (row >= mrows) continue;                            // rows that do not exist leave what is there: their results are not stored
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < P; ++c) {
      float h[8];
      unpack8<T>(x[i][c], h);
      if (a.residual) {
        float r[8];
        unpack8<T>(res[i][c], r);
#pragma unroll
        for (int e = 0; e < 8; ++e) h[e] = to_float(from_float<T>(h[e] + r[e]));       // the sum lives in T
        x[i][c] = pack8<T>(h);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = ss + h[e] * h[e];
    }
    if (a.residual_out && (int)blockIdx.x == row) {
      T* hp = reinterpret_cast<T*>(a.residual_out) + (int64_t)(m0 + row) * K + 8 * lane;
#pragma unroll
      for (int c = 0; c < P; ++c) *reinterpret_cast<uint4*>(hp + 512 * c) = x[i][c];
    }
    const SharedDivisor denom(sqrtf(four_rows_sum(row16_sum(ss)) / (float)K + a.eps));
    char* place = lds + r8 * kPanel + i * 1024 + wave * 128 + (((lane & 7) ^ wave) << 4);
#pragma unroll
    for (int c = 0; c < P; ++c) {
      float h[8];
      unpack8<T>(x[i][c], h);
      const float g[8] = {gam[c][0].x, gam[c][0].y, gam[c][0].z, gam[c][0].w, gam[c][1].x, gam[c][1].y, gam[c][1].z, gam[c][1].w};
#pragma unroll
      for (int e = 0; e < 8; ++e) h[e] = denom.divide(h[e]) * g[e];
      *reinterpret_cast<uint4*>(place + 8 * kPanel * c) = pack8<T>(h);
    }
  }
  __syncthreads();
  // ---- products: panels wave * P .. of x, the wave's weights through its own place (a wave's LDS accesses stay in order) ----
  v4f acc[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) acc[ct] = (v4f){0.f, 0.f, 0.f, 0.f};
  char* own = lds + kX + wave * CT * kPanel;
  const int frag = ((lane >> 3) & 1) * 1024 + (lane & 7) * 128, p0 = ((lane >> 4) ^ (lane & 7)) << 4;
#pragma unroll
  for (int p = 0; p < P; ++p) {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        *reinterpret_cast<uint4*>(own + ct * kPanel + b * 1024 + r8 * 128 + (((lane & 7) ^ r8) << 4)) = w[p][ct][b];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const uint4 xf = *reinterpret_cast<const uint4*>(lds + (wave * P + p) * kPanel + frag + (p0 ^ (64 * kk)));
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
        acc[ct] = mfma16x16x32<T>(*reinterpret_cast<const uint4*>(own + ct * kPanel + frag + (p0 ^ (64 * kk))), xf, acc[ct]);
    }
    __builtin_amdgcn_wave_barrier();
  }
  float4* part = reinterpret_cast<float4*>(lds + kX);      // the wave's own place again: CT KB of CT * 2
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) part[(2 * wave * CT + ct) * 64 + lane] = make_float4(acc[ct][0], acc[ct][1], acc[ct][2], acc[ct][3]);
  __syncthreads();
  if (wave >= CT) return;
  float s[4] = {0.f, 0.f, 0.f, 0.f}, up[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < W; ++k) {
    const float4 q = part[(2 * k * CT + wave) * 64 + lane];
    s[0] += q.x; s[1] += q.y; s[2] += q.z; s[3] += q.w;
  }
  const int cls = lane >> 4, m = lane & 15;
  if constexpr (GLU) {
#pragma unroll
    for (int r = 0; r < 4; ++r) up[r] = __shfl_xor(s[r], 32, 64);
    if (cls >= 2) return;
  }
  finish_four<T, GLU>(a, m < mrows ? m0 + m : a.M, first + (GLU ? 8 : 16) * wave + 4 * cls, s, up);
}

// ---- which kernel ----
// linear_rows_kernel up to here: from then on its lanes' different rows of x cost more than the ring's detour through LDS.  us at 1 / 3 / 4 rows,
// in registers against through the ring: 6144 x 4096 10.9 / 11.8 / 12.8 against 13.9, 2048 x 6144 6.8 / 7.2 / 7.5 against 10.0, 4096 x 12288 18.7 /
// 20.7 / 22.6 against 19.6, 24576 x 4096 33.7 / 34.5 / 35.0 against 35.4.
constexpr int kFewRows = 3;
constexpr int64_t kStreamBytes = 12 << 20;                 // weights from this size on are marked as read once (see linear_ring_kernel)

// Columns per workgroup of the ring form: the narrowest tile with which the copies of a CU (its workgroups one after the other,
// each bringing `columns + rows` rows of K values, at the 30 B per clock measured for such copies) take no longer than the weights take from
// HBM, N / 100 in these units; else the tile with which they take the least.  us at 64 rows with 16 / 32 / 64 / 96 columns: 4096 x 4096 13.3 / 15.8 / 21.1 / 33,
// 6144 x 4096 22.3 / 17.2 / 22.0 / 34, 12288 x 2048 22 / 19.2 / 15.4 / 18.8, 24576 x 4096 75 / 53.8 / 53 / 44.2.
static int ring_columns(int M, int N) {
  if (N <= 4096) return 16;
  const int rows = (M + 15) / 16 * 16, widths[3] = {32, 64, 96};
  int best = 0, best_cost = 0;
  for (int c : widths) {
    const int cost = ((N + c - 1) / c + 255) / 256 * (c + rows);
    if (cost * 100 <= N) return c;
    if (!best || cost < best_cost) { best = c; best_cost = cost; }
  }
  return best;
}

// Splits of K: with narrow tiles every workgroup reads all of x, rows * K values, and the CUs' copies of it, not the weights, take the time
// once K is long; with wider tiles and three or four splits of K the workgroups are as many and each reads a part of x, for
// a second launch (2.5 us) that adds the partial sums up.  us at 16 / 33 / 64 rows, whole and split: 4096 x 12288 22.1 / 30.7 / 37.1 and
// 21.1 / 23.0 / 27.0, 5120 x 8192 23.6 / 27.6 / 32.0 and 20.5 / 21.4 / 24.5, 4096 x 6144 12.9 / 17.6 / 20.9 and 13.0 / 14.4 / 17.4,
// 2048 x 6144 10.0 / 13.9 / 18.0 and 8.6 / 9.7 / 11.7, 1024 x 6144 9.2 / 13.3 / 17.2 and 6.8 / 8.5 / 9.6.  No gain: 4 to 24 rows of 2736 to 4096
// columns and K of 6144 to 8192 (3072 x 8192 at 16 rows 13.8 and 14.8), 4096 x 4096 (13.6 and 13.2 at 64 rows), more columns
// (6144 x 4096 18.5 and 18.3), 1024 x 3072 up to 32 rows (5.4 and 6.2 at 16; 9.0 and 7.4 at 64).
static LinearSplit linear_split(int M, int N, int K) {
  constexpr int kTiles = 256 / 3;                           // at most so many, for three splits of each over 256 CUs
  if (M <= kFewRows || N < 1024 || N > 64 * kTiles) return {0, 1};
  const bool narrow = N <= 2048, many = M > 32;
  if (!(K >= 12288 || (K >= 6144 && (narrow || N > 4096 || many)) || (K >= 3072 && narrow && many))) return {0, 1};
  const int columns = N <= 16 * kTiles ? 16 : N <= 32 * kTiles ? 32 : 64;
  const int splits = 256 / ((N + columns - 1) / columns);
  return {columns, splits < 4 ? splits : 4};
}

// The same where the residual norm follows and its launch adds the parts up (parts_norm_kernel): it reads 4 bytes a part instead of two, and has
// less to wait for than the norm alone, a thread for four numbers.  So parts pay nearly everywhere: two to four of them, with the narrowest
// tile of which 256 CUs have a workgroup each, of at least two stages but for a last part (K of 2560, up to 1024 columns: 3, 3, 3
// and 1).  us with the norm at 4 / 17 / 40 / 61 rows, apart (linear_split's
// where it takes the shape) and now: 1024 x 2048 6.8 / 7.0 / 7.2 / 7.4 and 5.4 / 5.9 / 6.1 / 6.6, 1024 x 3072 7.4 / 7.3 / 9.8 / 10.4 and 5.7 / 6.2 / 6.5 / 7.1,
// 2048 x 2048 6.8 / 7.0 / 8.2 / 9.0 and 6.1 / 6.6 / 7.1 / 7.8, 2048 x 6144 10.5 / 11.3 / 12.8 / 14.1 and 8.3 / 9.1 / 10.5 / 11.8, 2560 x 2560 8.7 / 9.7 / 11.7 / 12.8
// and 7.3 / 7.7 / 8.8 / 10.2, 4096 x 4096 10.9 / 12.0 / 14.3 / 16.3 and 10.2 / 11.0 / 12.5 / 14.0, 4096 x 12288 23.5 / 23.4 / 25.7 / 28.4 and 20.7 / 21.5 / 23.5 / 25.9,
// 5120 x 5120 19.1 / 18.1 / 21.6 / 25.5 and 13.8 / 14.8 / 16.9 / 19.0, 7168 x 2048 12.2 / 12.2 / 13.9 / 15.1 and 10.7 / 11.3 / 12.7 / 14.3; least: 4096 x 1024
// 7.1 / 7.6 / 8.0 / 8.5 and 6.7 / 7.0 / 7.7 / 8.3, 2048 x 1024 5.9 / 6.0 / 6.9 / 7.3 and 5.6 / 6.0 / 6.7 / 7.2.  Past that none: 8192 x 4096 17.9 / 17.2 / 19.9 / 22.0
// and 17.7 / 18.4 / 19.8 / 21.3.  Up to 4096 columns two parts of 32 or four of 64 fill the chip: 4096 x 2048 7.7 / 8.3 / 9.4 / 10.4 and 8.0 / 8.7 / 10.0 / 11.3, 3072 x 3072
// 8.3 / 8.9 / 10.3 / 11.5 and 8.4 / 9.1 / 10.2 / 11.5, 4096 x 12288 21.8 / 21.7 / 25.1 / 29.0 and as above.
static LinearSplit linear_norm_split(int M, int N, int K) {
  if (M <= kFewRows || N < 512 || N > 7168 || K < (N > 4096 ? 2048 : 1024)) return {0, 1};
  if (N <= 1024) return {K < 2048 ? 32 : 16, 4};
  if (N <= 2048) return {32, 4};
  if (N <= 2720) return {32, 3};
  if (N <= 4096) return K < 4096 ? LinearSplit{32, 2} : LinearSplit{64, 4};
  return {64, N <= 5440 ? 3 : 2};
}

// Few columns leave CUs without a workgroup, and each one with all the rows copies `rows + 16` rows of K values one stage after the other: the tiles of
// 16 rows as workgroups of their own read the weights once each, from the L2 after the first, and copy 32 rows.  While they find a CU each: past
// 256 the second round costs more than the rows.  us whole / apart: 49 x 512 x 14336 34.5 / 16.0, 64 x 512 x 4096 10.0 / 5.8, 17 x 2048 x 4096
// (256 workgroups) 8.4 / 7.4, 64 x 1024 x 4096 gated (256) 10.7 / 6.8; 33 x 2048 x 14336 gated (384) 29.2 / 36.4, 17 x 2720 x 4096 (340)
// 9.0 / 12.7.  A long K with 1024 columns on is cut into parts instead where the caller brings the room (64 x 1024 x 14336 15.7, apart 19.3).
static bool rows_apart(int M, int N) { return (N + 15) / 16 * ((M + 15) / 16) <= 256; }

template <typename T, bool GLU>
static int launch_rows(const LinearArgs& a, hipStream_t stream) {
  // few columns: narrow tiles and more waves on a tile's K, to have more loads under way.  us at one row with 8 columns and 8 / 4 waves, 16 columns
  // and 4 waves: 1024 x 3072 4.0 / 4.1 / 5.2, 4096 x 4096 7.7 / 7.3 / 7.9, 12288 x 2048 - / 11 / 10.8.  The order of a sum follows
  // from the number of waves: it does not depend on GLU.
  constexpr int WT = GLU ? 2 : 1;
  const auto grid = [&](int wt) { const int c = wt * (GLU ? 4 : 8); return dim3((unsigned)(((GLU ? a.N / 2 : a.N) + c - 1) / c)); };
  if (a.N <= 2048) {
    if (a.K % 1024 == 0) linear_rows_kernel<T, WT, 2, 8, GLU><<<grid(WT), dim3(512), 0, stream>>>(a);
    else linear_rows_kernel<T, WT, 1, 8, GLU><<<grid(WT), dim3(512), 0, stream>>>(a);
  } else if (a.N <= 8192) {
    linear_rows_kernel<T, WT, 2, 4, GLU><<<grid(WT), dim3(256), 0, stream>>>(a);
  } else {
    linear_rows_kernel<T, 2, 2, 4, GLU><<<grid(2), dim3(256), 0, stream>>>(a);
  }
  return launch_status();
}

template <typename T, int MT, bool GLU>
static int launch_ring(LinearArgs a, hipStream_t stream) {
  const bool stream_weights = (int64_t)a.N * a.K * 2 >= kStreamBytes;
  const LinearSplit split = a.part ? a.split : LinearSplit{ring_columns(a.M, a.N), 1};
  const int columns = split.columns, steps = a.K / (columns == 16 ? 256 : 128);
  a.part_steps = (steps + split.splits - 1) / split.splits;
  const dim3 grid((unsigned)((a.N + columns - 1) / columns), (unsigned)split.splits, (unsigned)((a.M + 16 * MT - 1) / (16 * MT)));
  constexpr int S = MT > 2 ? 3 : 4;
  switch (columns) {
    case 16:
      if (stream_weights) linear_ring_kernel<T, MT, 1, 4, 1, S, true, GLU><<<grid, dim3(256), 0, stream>>>(a);
      else linear_ring_kernel<T, MT, 1, 4, 1, S, false, GLU><<<grid, dim3(256), 0, stream>>>(a);
      break;
    case 32:
      if (stream_weights) linear_ring_kernel<T, MT, 1, 2, 2, 4, true, GLU><<<grid, dim3(256), 0, stream>>>(a);
      else linear_ring_kernel<T, MT, 1, 2, 2, 4, false, GLU><<<grid, dim3(256), 0, stream>>>(a);
      break;
    case 64: linear_ring_kernel<T, MT, 2, 2, 2, 3, true, GLU><<<grid, dim3(256), 0, stream>>>(a); break;
    default: linear_ring_kernel<T, MT, 3, 2, 2, 4, true, GLU><<<grid, dim3(256), 0, stream>>>(a);
  }
  const int status = launch_status();
  if (status != MVLLM_OK || !a.part || a.leave_parts) return status;
  linear_sum_kernel<T><<<dim3((unsigned)(((int64_t)a.M * a.N / 4 + 255) / 256)), dim3(256), 0, stream>>>(a, split.splits);
  return launch_status();
}

template <typename T, bool GLU>
static int launch_plain(const LinearArgs& a, hipStream_t stream) {
  if (a.M <= kFewRows) return launch_rows<T, GLU>(a, stream);
  if (((int64_t)(a.M - 1) * a.x_row_stride + a.K) * 2 > 0xffffffffll) {      // past a buffer descriptor's offsets: kFewRows at a time
    LinearArgs part = a;
    for (int m = 0; m < a.M; m += kFewRows) {
      part.x = reinterpret_cast<const T*>(a.x) + (int64_t)m * a.x_row_stride;
      part.out = reinterpret_cast<T*>(a.out) + (int64_t)m * (GLU ? a.N / 2 : a.N);
      part.M = a.M - m < kFewRows ? a.M - m : kFewRows;
      const int bad = launch_rows<T, GLU>(part, stream);
      if (bad) return bad;
    }
    return MVLLM_OK;
  }
  if (a.M <= 16 || (!a.part && rows_apart(a.M, a.N))) return launch_ring<T, 1, GLU>(a, stream);
  if (a.M <= 32) return launch_ring<T, 2, GLU>(a, stream);
  if (a.M <= 48) return launch_ring<T, 3, GLU>(a, stream);
  return launch_ring<T, 4, GLU>(a, stream);
}

// Shapes the norm form takes: K of 512, 1024 or 2048 (512 P), at least as many column tiles as rows of a row tile.  The number reported for a shape
// is the split of K that defined the set: the fewest waves that give 1024 of them in all with one burst of 128 or 256 values
// each; 0 when there is none.
static bool norm_fits(int W, int steps) { return steps == 4 || (steps == 8 && W <= 8); }
static int norm_row_tiles(int M) { return (M + 15) / 16; }
static int norm_waves(int tiles, int K) {
  int best = 0;
  for (int w = 4; w <= 16; w *= 2) {
    if (K % (32 * w) != 0 || !norm_fits(w, K / w / 32)) continue;
    best = w;
    if ((int64_t)tiles * w >= 1024) break;
  }
  return best;
}
static bool norm_takes(int M, int N, int K) {
  return norm_waves(N / 16 * norm_row_tiles(M), K) != 0 && N / 16 >= (M < 16 ? M : 16);
}

template <typename T, int P, bool GLU>
static int launch_norm(const LinearArgs& a, hipStream_t stream) {
  // 32 columns halve what the rows cost where 16 would give a CU more than one workgroup
  const int wide = a.N > 4096;
  const dim3 grid((unsigned)((a.N + (wide ? 31 : 15)) / (wide ? 32 : 16)), (unsigned)a.row_tiles);
  if (wide) linear_norm_kernel<T, 2, P, GLU><<<grid, dim3(512), 0, stream>>>(a);
  else linear_norm_kernel<T, 1, P, GLU><<<grid, dim3(512), 0, stream>>>(a);
  return launch_status();
}

template <typename T, bool GLU>
static int launch_norm_k(const LinearArgs& a, hipStream_t stream) {
  if (!norm_takes(a.M, a.N, a.K)) return MVLLM_ERR_UNSUPPORTED;
  switch (a.K) {
    case 512: return launch_norm<T, 1, GLU>(a, stream);
    case 1024: return launch_norm<T, 2, GLU>(a, stream);
    case 2048: return launch_norm<T, 4, GLU>(a, stream);
    default: return MVLLM_ERR_UNSUPPORTED;
  }
}

template <typename T>
static int launch_linear_fused(const LinearArgs& a, bool glu, hipStream_t stream) {
  if (a.gamma) return glu ? launch_norm_k<T, true>(a, stream) : launch_norm_k<T, false>(a, stream);
  return glu ? launch_plain<T, true>(a, stream) : launch_plain<T, false>(a, stream);
}

static int linear_check(const void* out, const void* x, const void* w, const void* bias, int64_t x_row_stride, int M,
                        int N, int K, int dtype) {
  if (dtype != MVLLM_BF16 && dtype != MVLLM_F16) return dtype_size(dtype) == 0 ? MVLLM_ERR_BAD_DTYPE : MVLLM_ERR_UNSUPPORTED;
  if (M < 0 || N <= 0 || K <= 0 || x_row_stride < K) return MVLLM_ERR_BAD_SHAPE;
  if (M == 0) return MVLLM_OK;
  if (!out || !x || !w) return MVLLM_ERR_NULL_POINTER;
  if (M > 64 || N % 16 != 0 || K % 512 != 0 || x_row_stride % 8 != 0) return MVLLM_ERR_UNSUPPORTED;
  if (!aligned16(x) || !aligned16(w) || (reinterpret_cast<uintptr_t>(out) & 7u) || (reinterpret_cast<uintptr_t>(bias) & 7u))
    return MVLLM_ERR_MISALIGNED;
  return MVLLM_OK;
}

}  // namespace mvllm

using namespace mvllm;

static int linear_plain(void* out, const void* x, const void* w, const void* bias, int64_t x_row_stride, int M, int N, int K,
                        int gelu, int dtype, void* stream, float* part = nullptr) {
  const int bad = linear_check(out, x, w, bias, x_row_stride, M, N, K, dtype);
  if (bad || M == 0) return bad;
  LinearArgs a{};
  a.out = out; a.x = x; a.w = w; a.bias = bias; a.x_row_stride = x_row_stride; a.M = M; a.N = N; a.K = K;
  a.gelu = gelu; a.part = part;
  if (part) a.split = linear_split(M, N, K);
  return dtype == MVLLM_BF16 ? launch_linear_fused<bf16_t>(a, false, (hipStream_t)stream)
                             : launch_linear_fused<f16_t>(a, false, (hipStream_t)stream);
}

extern "C" int mvllm_linear_small_m(void* out, const void* x, const void* w, const void* bias, int64_t x_row_stride,
                                    int M, int N, int K, int dtype, void* stream) {
  return linear_plain(out, x, w, bias, x_row_stride, M, N, K, 0, dtype, stream);
}

extern "C" int mvllm_linear_small_m_gelu(void* out, const void* x, const void* w, const void* bias, int64_t x_row_stride,
                                         int M, int N, int K, int dtype, void* stream) {
  return linear_plain(out, x, w, bias, x_row_stride, M, N, K, 1, dtype, stream);
}

extern "C" size_t mvllm_linear_small_m_split_bytes(int M, int N, int K, int64_t x_row_stride) {
  if (M <= 0 || M > 64 || N <= 0 || N % 16 != 0 || K <= 0 || K % 512 != 0 || ((int64_t)(M - 1) * x_row_stride + K) * 2 > 0xffffffffll) return 0;
  const int splits = linear_split(M, N, K).splits;
  return splits < 2 ? 0 : (size_t)splits * M * N * sizeof(float);
}

extern "C" int mvllm_linear_small_m_split(void* out, const void* x, const void* w, const void* bias, int64_t x_row_stride,
                                          int M, int N, int K, int gelu, int dtype, void* workspace, size_t workspace_bytes, void* stream) {
  const size_t need = mvllm_linear_small_m_split_bytes(M, N, K, x_row_stride);
  if (need != 0 && (!workspace || !aligned16(workspace) || workspace_bytes < need)) return MVLLM_ERR_WORKSPACE;
  return linear_plain(out, x, w, bias, x_row_stride, M, N, K, gelu != 0, dtype, stream, need != 0 ? reinterpret_cast<float*>(workspace) : nullptr);
}

extern "C" int mvllm_linear_small_m_plan(int M, int N, int K, int norm, int glu, int dtype, int* waves) {
  if (dtype != MVLLM_BF16 && dtype != MVLLM_F16) return dtype_size(dtype) == 0 ? MVLLM_ERR_BAD_DTYPE : MVLLM_ERR_UNSUPPORTED;
  if (M <= 0 || N <= 0 || K <= 0) return MVLLM_ERR_BAD_SHAPE;
  if (M > 64 || N % 16 != 0 || K % 512 != 0 || (glu && N % 32 != 0)) return MVLLM_ERR_UNSUPPORTED;
  int w = M <= kFewRows && N <= 2048 ? 8 : 4;
  if (norm) {
    if (!norm_takes(M, N, K)) return MVLLM_ERR_UNSUPPORTED;
    w = norm_waves(N / 16 * norm_row_tiles(M), K);
  }
  if (waves) *waves = w;
  return MVLLM_OK;
}

extern "C" int mvllm_norm_linear_small_m(void* out, void* residual_out, const void* x, const void* residual,
                                         const float* gamma, float eps, const void* w, const void* bias,
                                         int64_t x_row_stride, int M, int N, int K, int glu, int dtype, void* stream) {
  const int bad = linear_check(out, x, w, bias, x_row_stride, M, N, K, dtype);
  if (bad || M == 0) return bad;
  if (glu && N % 32 != 0) return MVLLM_ERR_UNSUPPORTED;
  if ((residual || residual_out) && !gamma) return MVLLM_ERR_NULL_POINTER;
  if (gamma) {
    if (!aligned16(gamma) || (residual && !aligned16(residual)) || (residual_out && !aligned16(residual_out)))
      return MVLLM_ERR_MISALIGNED;
    if (residual_out && (residual_out == x || residual_out == residual)) return MVLLM_ERR_BAD_SHAPE;
  }
  LinearArgs a{};
  a.out = out; a.x = x; a.w = w; a.bias = bias; a.x_row_stride = x_row_stride; a.M = M; a.N = N; a.K = K;
  a.residual = residual; a.residual_out = residual_out; a.gamma = gamma; a.eps = eps;
  a.row_tiles = norm_row_tiles(M);
  return dtype == MVLLM_BF16 ? launch_linear_fused<bf16_t>(a, glu != 0, (hipStream_t)stream)
                             : launch_linear_fused<f16_t>(a, glu != 0, (hipStream_t)stream);
}

extern "C" size_t mvllm_linear_add_rms_norm_bytes(int M, int N, int K, int64_t x_row_stride) {
  if (M <= 0 || M > 64 || N <= 0 || N % 16 != 0 || K <= 0 || K % 512 != 0 || ((int64_t)(M - 1) * x_row_stride + K) * 2 > 0xffffffffll) return 0;
  const int splits = linear_norm_split(M, N, K).splits;
  return splits < 2 ? 0 : (size_t)splits * M * N * sizeof(float);
}

extern "C" int mvllm_linear_add_rms_norm(void* out, void* residual_out, const void* x, const void* w, const void* bias, const void* residual,
                                         const float* gamma, float eps, int64_t x_row_stride, int M, int N, int K, int dtype, void* workspace,
                                         size_t workspace_bytes, void* stream) {
  const int bad = linear_check(out, x, w, bias, x_row_stride, M, N, K, dtype);
  if (bad || M == 0) return bad;
  if (!residual_out || !residual || !gamma) return MVLLM_ERR_NULL_POINTER;
  if (!aligned16(out) || !aligned16(residual_out) || !aligned16(residual) || !aligned16(gamma)) return MVLLM_ERR_MISALIGNED;
  const size_t need = mvllm_linear_add_rms_norm_bytes(M, N, K, x_row_stride);
  if (need == 0) return MVLLM_ERR_UNSUPPORTED;
  if (!workspace || !aligned16(workspace) || workspace_bytes < need) return MVLLM_ERR_WORKSPACE;
  LinearArgs a{};
  a.x = x; a.w = w; a.x_row_stride = x_row_stride; a.M = M; a.N = N; a.K = K;
  a.part = reinterpret_cast<float*>(workspace); a.split = linear_norm_split(M, N, K); a.leave_parts = true;
  const int status = dtype == MVLLM_BF16 ? launch_linear_fused<bf16_t>(a, false, (hipStream_t)stream)
                                         : launch_linear_fused<f16_t>(a, false, (hipStream_t)stream);
  if (status != MVLLM_OK) return status;
  return launch_parts_norm(out, residual_out, a.part, a.split.splits, bias, residual, gamma, eps, M, N, dtype, (hipStream_t)stream);
}
