// Mixture of experts: the router's choice, the rows sorted by expert, and the experts' products.
//   moe_route   scores s = sigmoid(z), choice scores s + correction; groups of neighbouring experts by the sum of their two
//               largest choice scores, the best `keep` groups stay open; the `top` largest choice scores of those are chosen,
//               weights s / (sum of the chosen s + 1e-20); or s = softmax(z), the weights s as they are; the last outputs may
//               stand for no expert but for the input itself: their id is -1
//   moe_plan    (token, choice) pairs sorted by expert, and tiles of 64, 128 or 256 sorted rows per expert
//   moe_linear  out[row] = x[row] W_e^T, optionally silu(gate) * up or its clamped form behind it: W_e [2 F, K] with gate and up rows in turns of
//               32, so that both halves of an output are in one lane
// Products, by the number of rows: very few (no plan; a workgroup finds its expert's rows itself, its waves share K), many (bf16: tiles of 32 x 64, 64 x 64, 64 x 128,
// 128 x 128 or 256 x 256 on the matrix unit over sorted rows), any (fp32, over sorted rows).
#include "expert_tiles.h"
#include "prefill_tiles.h"
#include <cmath>

#pragma clang fp contract(off)

namespace mvllm {

// ---- routing ----
struct RouteArgs {
  int32_t* ids;            // [T, top]
  float* weights;          // [T, top]
  const float* z;          // [T, z_stride] logits
  const float* correction; // [E] or null
  int64_t z_stride;
  int rows, experts, top, groups, keep;
  int identity;            // of the experts: the last ones, whose output is their input
  bool softmax, renormalize;
};

// One token per wave; lane l has experts l, l + 64, ...
template <int NE>
__global__ __launch_bounds__(256) void moe_route_kernel(const RouteArgs a) {
  __shared__ float choice_of[4][64 * NE], group_of[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = blockIdx.x * 4 + wave;
  const bool live = row < a.rows;
  const int E = a.experts;
  float s[NE], choice[NE];
#pragma unroll
  for (int i = 0; i < NE; ++i) {
    const int e = lane + 64 * i;
    s[i] = 0.f;
    choice[i] = -INFINITY;
    if (live && e < E) {
      const float z = a.z[(int64_t)row * a.z_stride + e];
      s[i] = a.softmax ? z : 1.0f / (1.0f + expf(-z));
    }
  }
  if (a.softmax) {
    float most = -INFINITY, sum = 0.f;
#pragma unroll
    for (int i = 0; i < NE; ++i) most = fmaxf(most, lane + 64 * i < E ? s[i] : -INFINITY);
    most = wave_max_in_registers(most);
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      s[i] = lane + 64 * i < E ? expf(s[i] - most) : 0.f;
      sum += s[i];
    }
    sum = four_rows_sum(row16_sum(sum));
#pragma unroll
    for (int i = 0; i < NE; ++i) s[i] /= sum;
  }
#pragma unroll
  for (int i = 0; i < NE; ++i) {
    const int e = lane + 64 * i;
    if (live && e < E) choice[i] = s[i] + (a.correction ? a.correction[e] : 0.f);
    choice_of[wave][e] = choice[i];
  }
  if (a.groups > 1) {
    const int size = E / a.groups;
    __syncthreads();
    if (lane < a.groups) {
      float first = -INFINITY, second = -INFINITY;
      for (int j = 0; j < size; ++j) {
        const float x = choice_of[wave][lane * size + j];
        second = fmaxf(second, fminf(first, x));
        first = fmaxf(first, x);
      }
      group_of[wave][lane] = size > 1 ? first + second : first;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int e = lane + 64 * i;
      if (e >= E) continue;
      const int g = e / size;
      const float mine = group_of[wave][g];
      int before = 0;
      for (int j = 0; j < a.groups; ++j) {
        const float x = group_of[wave][j];
        before += x > mine || (x == mine && j < g);
      }
      if (before >= a.keep) choice[i] = -INFINITY;
    }
  }
  float my_s = 0.f, sum = 0.f;
  int my_id = 0;
  for (int k = 0; k < a.top; ++k) {
    float mine = choice[0];
#pragma unroll
    for (int i = 1; i < NE; ++i) mine = fmaxf(mine, choice[i]);
    const float best = wave_max_in_registers(mine);
    int id = -1;                                    // the first expert that has it
    float best_s = 0.f;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const unsigned long long at = __ballot(choice[i] == best);
      if (id < 0 && at != 0ull) {
        const int l = __builtin_amdgcn_readfirstlane(__builtin_ctzll(at));
        id = 64 * i + l;
        best_s = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(s[i]), l));
        if (lane == l) choice[i] = -INFINITY;
      }
    }
    if (id < 0 || id >= E) id = 0;                  // (nothing left to choose)
    sum += best_s;
    if (lane == k) { my_s = best_s; my_id = id; }
  }
  if (live && lane < a.top) {
    a.ids[(int64_t)row * a.top + lane] = my_id < E - a.identity ? my_id : -1;
    a.weights[(int64_t)row * a.top + lane] = a.renormalize ? my_s / (sum + 1e-20f) : my_s;
  }
}

// ---- pairs sorted by expert ----
constexpr int kPlanPairs = 2048, kMaxExperts = 1024;
constexpr int kLargeTileRows = 384;      // rows per expert from which tiles are large
// ... up to which they are small: at 47 per expert (500 rows, top 6 of 64, width 2048) 76 + 42 us against 98 + 44 as tiles of 128, at
// 65 121 + 73 against 100 + 48: experts of two tiles read their weights twice.
constexpr int kSmallTileRows = 48;
// An expert's last large tile is apart from the others up to here: it is short and brings the chip's last round to an end.  With more rows it takes
// its time and would read the weights again, which the expert's other tiles have in the L2.  us as all that are not whole, up to 64 rows,
// none apart: 64 experts, 400 rows each, 1536 x 2048 203 / 182 / 180, of 896 x 2240 288 / 254 / 255; 768 350 / 307 / 337 and 688 / 629 / 669; the 8192 rows of
// a mixture, top 6 of 64, routed unevenly, 820 / 802 / 827.
constexpr int kApartRows = 64;
// ... where there are rounds enough: with few tiles all run at once, and an expert's do so on one XCD (8 experts of 600 rows, 320 x 1536, 33.9 us none
// apart and 35.7).
constexpr int kApartPairs = 8192;

struct PlanArgs {
  const int32_t* ids;      // [pairs]
  int32_t* hist;           // [blocks, E]
  int32_t* sorted_pair;    // [pairs]: pair at a sorted place
  int32_t* place;          // [pairs]: sorted place of a pair
  int32_t* row_start;      // [E + 1]
  struct Tiles {
    int32_t* expert;       // [max tiles]
    int32_t* row;          // [max tiles]: first sorted row
    int32_t* num;          // [2] those in order, those behind them (see find_tile)
  } tiles[2];              // of tile_rows; and, where that is 128, of 256
  int pairs, experts, blocks, tile_rows;
};

__global__ __launch_bounds__(256) void moe_count_kernel(const PlanArgs a) {
  __shared__ int32_t count[kMaxExperts];
  for (int e = threadIdx.x; e < a.experts; e += 256) count[e] = 0;
  __syncthreads();
  const int end = min((int)(blockIdx.x + 1) * kPlanPairs, a.pairs);
  for (int p = blockIdx.x * kPlanPairs + threadIdx.x; p < end; p += 256) {
    const int id = a.ids[p];
    if (id >= 0) atomicAdd(&count[id], 1);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < a.experts; e += 256) a.hist[(int64_t)blockIdx.x * a.experts + e] = count[e];
}

// A chain of latencies, not bytes: the counts of the blocks, sums over the experts, places.  With the counts' loads one by one and the sums in ten rounds
// with two barriers each 14 us at 49152 pairs of 64 experts, so 5.9; 1800 pairs 5.1 and 3.5.
// kRows: a.tile_rows.  It has no more sums than its tiles need: five of them for every plan took a small one 0.5 us.
template <int kRows>
__global__ __launch_bounds__(1024) void moe_place_kernel(const PlanArgs a) {
  constexpr bool large = kRows == 256, both = kRows == 128;
  constexpr int kSums = both ? 4 : large ? 3 : 2;   // rows; tiles in order; of the tiling of 256 rows, those and the ones behind them
  __shared__ int32_t sum_to[kSums][kMaxExperts + 1], cursor[kMaxExperts], of_wave[kSums][16];
  const int e = threadIdx.x;
  int n = 0, mine = 0;
  if (a.blocks == 1) {                              // counted here
    cursor[e] = 0;
    __syncthreads();
    for (int p = e; p < a.pairs; p += 1024) {
      const int id = a.ids[p];
      if (id >= 0) atomicAdd(&cursor[id], 1);
    }
    __syncthreads();
    n = cursor[e];
    __syncthreads();
  } else if (e < a.experts) {
#pragma unroll 8
    for (int b = 0; b < a.blocks; ++b) {            // (loads of several blocks under way)
      const int of_block = a.hist[(int64_t)b * a.experts + e];
      mine += b < (int)blockIdx.x ? of_block : 0;
      n += of_block;
    }
  }
  // inclusive sums over the experts: within a wave, then over the waves before it
  const bool apart = (large || both) && n % 256 != 0 && n % 256 <= kApartRows && a.pairs >= kApartPairs;      // the last tile of 256 goes behind all others
  int sums[kSums];
  sums[0] = n;
  sums[1] = (n + kRows - 1) / kRows - (large && apart);
  if constexpr (both) sums[2] = (n + 255) / 256 - apart;
  if constexpr (large || both) sums[kSums - 1] = apart;
  const int lane = e & 63, wave = __builtin_amdgcn_readfirstlane(e >> 6);
  const bool some = 64 * wave < a.experts;
  if (some) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
#pragma unroll
      for (int i = 0; i < kSums; ++i) {
        const int before = __shfl_up(sums[i], o, 64);
        sums[i] += lane >= o ? before : 0;
      }
    if (lane == 63)
      for (int i = 0; i < kSums; ++i) of_wave[i][wave] = sums[i];
  }
  __syncthreads();
  if (some) {
    for (int w = 0; w < wave; ++w)
#pragma unroll
      for (int i = 0; i < kSums; ++i) sums[i] += of_wave[i][w];
#pragma unroll
    for (int i = 0; i < kSums; ++i) sum_to[i][e + 1] = sums[i];
  }
  if (e < kSums) sum_to[e][0] = 0;
  __syncthreads();
  const int32_t* total = sum_to[0];
  if (e < a.experts) cursor[e] = total[e] + mine;
  __syncthreads();
  const int end = min((int)(blockIdx.x + 1) * kPlanPairs, a.pairs);
  for (int p = blockIdx.x * kPlanPairs + threadIdx.x; p < end; p += 1024) {
    const int id = a.ids[p];
    if (id < 0) {                                   // no expert's: nobody computes or reads it
      a.place[p] = -1;
      continue;
    }
    const int at = atomicAdd(&cursor[id], 1);
    a.sorted_pair[at] = p;
    a.place[p] = at;
  }
  if (blockIdx.x == 0 && e < a.experts) {
    a.row_start[e] = total[e];
    if (e == a.experts - 1) a.row_start[e + 1] = total[e + 1];
#pragma unroll
    for (int i = 0; i < 1 + both; ++i) {
      const PlanArgs::Tiles& t = a.tiles[i];
      const bool wide = large || i == 1;
      const int32_t *tiles = sum_to[1 + i], *parts = sum_to[kSums - 1];      // (parts: of the wide tiling alone)
      const int rows = i == 0 ? kRows : 256;
      if (e == a.experts - 1) {
        t.num[0] = tiles[e + 1];
        t.num[1] = wide ? parts[e + 1] : 0;
      }
      for (int k = tiles[e]; k < tiles[e + 1]; ++k) {
        t.expert[k] = e;
        t.row[k] = total[e] + (k - tiles[e]) * rows;
      }
      if (wide && parts[e + 1] > parts[e]) {
        const int k = tiles[a.experts] + parts[e];
        t.expert[k] = e;
        t.row[k] = total[e + 1] - n % 256;
      }
    }
  }
}

// ---- products ----
struct ExpertLinearArgs {
  void* out;                   // [pairs, out_stride]
  const void* x;               // [*, x_stride]
  const void* w;               // [E, N, K]
  const int32_t* ids;          // [pairs] (few)
  const int32_t* sorted_pair;  // (many, any) plan, see above
  const int32_t* row_start;
  const int32_t* tile_expert;
  const int32_t* tile_row;
  const int32_t* num_tiles;
  int64_t x_stride, out_stride;
  int pairs, experts, N, K;
  int per_token;               // > 0: pair p reads row p / per_token of x; 0: the row of its own (sorted) place
  int max_tiles, n_tiles;
  uint32_t x_bytes;            // (many) what x holds
  float alpha, limit, shift;   // of kClampedGlu
  int groups;                  // (large) workgroups per XCD
  uint32_t token_factor;       // (large) (2^32 - 1) / per_token
  // The product of an expert that all rows go through, as more tiles of the same launch: row r of x to row r of out.  On its own it took two or three
  // launches that leave CUs idle at their ends, and the activation between them went through memory as twice as many numbers.  us of a mixture and the norm
  // behind it, apart / so: 2048 wide, top 6 of 64 experts of 768 and 1536 shared, 3 rows 57 / 55, 100 137 / 120, 300 168 / 145, 1000 236 / 203, 8192 742 / 710;
  // 4096 wide, top 8 of 64 of 1280 and 2048 shared, 32 rows 328 / 317, 1000 621 / 572.
  struct Shared {
    const bf16_t* x;           // [rows, x_stride]
    const bf16_t* w;           // [N, K], with a gate all its rows before all of up's
    bf16_t* out;               // [rows, out_stride]
    int64_t x_stride, out_stride;
    int rows, N, K;            // (no rows: there is none)
    int row_tiles, n_tiles, blocks;     // (many) blocks: of the grid, in front of the others, a multiple of eight
    int units;                 // (large) what a tile takes, in tiles of the experts
    uint32_t x_bytes;
  } shared;
};

enum { kNoGlu = 0, kSiluGlu = 1, kClampedGlu = 2 };

// The row of the shared expert's weights for row r of a product's tiles, in which gate and up rows come in turns of 32.
template <int kGlu> __device__ __forceinline__ int shared_row(const ExpertLinearArgs& a, int r) {
  return kGlu != kNoGlu ? (r >> 6 << 5) + (r & 31) + ((r >> 5 & 1) != 0 ? a.shared.N / 2 : 0) : r;
}

// silu(g) * u, or with g' = min(g, limit) and u' = u within +-limit: g' sigmoid(alpha g') (u' + shift)
template <int kGlu> __device__ __forceinline__ float glu_of(const ExpertLinearArgs& a, float g, float u) {
  if constexpr (kGlu == kClampedGlu) {
    g = fminf(g, a.limit);
    return g * __builtin_amdgcn_rcpf(1.0f + __expf(-a.alpha * g)) * (fminf(fmaxf(u, -a.limit), a.limit) + a.shift);
  }
  return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * u;
}

// few: workgroup = (16 kTiles outputs, expert), its waves share K.  The rows of the expert are found in `ids`; rows are taken
// 16 at a time.
constexpr int kFewPairs = 512;

template <int kWaves, int kGlu, int kTiles>
__global__ __launch_bounds__(64 * kWaves) void moe_linear_few_kernel(const ExpertLinearArgs a) {
  constexpr int NT = kTiles * (kGlu ? 2 : 1);        // tiles of weight rows: with the gate, gate and up of an output tile in turn
  __shared__ uint16_t list[kFewPairs];
  __shared__ int found, count[kWaves];
  __shared__ float4 part[kWaves][NT][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, i16 = lane & 15;
  const int e = blockIdx.y;
  // the expert's pairs, in order: every wave looks through its share of the list, all loads at once
  constexpr int kEach = (kFewPairs + 64 * kWaves - 1) / (64 * kWaves);
  {
    const int share = (a.pairs + 64 * kWaves - 1) / (64 * kWaves) * 64, base = wave * share;
    int32_t id[kEach];
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
      const int p = base + 64 * i + lane;
      id[i] = 64 * i < share && p < a.pairs ? a.ids[p] : -1;
    }
    int n = 0;
#pragma unroll
    for (int i = 0; i < kEach; ++i) n += __popcll(__ballot(id[i] == e));
    if (lane == 0) count[wave] = n;
    __syncthreads();
    int at = 0, all = 0;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) {
      at += i < wave ? count[i] : 0;
      all += count[i];
    }
    if (tid == 0) found = all;
    if (all == 0) return;                           // (the same for every thread)
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
      const bool hit = id[i] == e;
      const unsigned long long hits = __ballot(hit);
      if (hit) list[at + __popcll(hits & ((1ull << lane) - 1))] = (uint16_t)(base + 64 * i + lane);
      at += __popcll(hits);
    }
  }
  __syncthreads();
  const int rows = found;
  const int n0 = blockIdx.x * 16 * kTiles;          // first output of the workgroup
  const bf16_t* w[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int out = kGlu ? n0 + 16 * (n / 2) : n0 + 16 * n;
    const int wr = kGlu ? (out >> 5) * 64 + (out & 31) + 32 * (n % 2) : out;
    w[n] = reinterpret_cast<const bf16_t*>(a.w) + ((int64_t)e * a.N + min(wr + i16, a.N - 1)) * a.K;
  }
  for (int r0 = 0; r0 < rows; r0 += 16) {
    const int pair = list[min(r0 + i16, rows - 1)];
    const bf16_t* x = reinterpret_cast<const bf16_t*>(a.x) + (int64_t)(a.per_token ? pair / a.per_token : pair) * a.x_stride;
    v4f acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int k0 = 64 * wave; k0 < a.K; k0 += 64 * kWaves) {            // a lane's 32 bytes: whole lines per row and wave
      const int k = k0 + 16 * g;
      uint4 xv[2], wv[NT][2];
#pragma unroll
      for (int half = 0; half < 2; ++half) {
#pragma unroll
        for (int n = 0; n < NT; ++n) wv[n][half] = load16_stream(w[n] + k + 8 * half);
        xv[half] = *reinterpret_cast<const uint4*>(x + k + 8 * half);
      }
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = mfma16x16x32<bf16_t>(wv[n][half], xv[half], acc[n]);
    }
    // lane: row i16, outputs 4 g + r
#pragma unroll
    for (int n = 0; n < NT; ++n) part[wave][n][lane] = make_float4(acc[n][0], acc[n][1], acc[n][2], acc[n][3]);
    __syncthreads();
    for (int m = wave; m < kTiles; m += kWaves) {   // output tile
      constexpr int kParts = kGlu ? 2 : 1;
      float z[kParts][4];
#pragma unroll
      for (int n = 0; n < kParts; ++n) {
        z[n][0] = z[n][1] = z[n][2] = z[n][3] = 0.f;
#pragma unroll
        for (int i = 0; i < kWaves; ++i) {
          const float4 p = part[i][m * kParts + n][lane];
          z[n][0] += p.x; z[n][1] += p.y; z[n][2] += p.z; z[n][3] += p.w;
        }
      }
      float o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = kGlu ? glu_of<kGlu>(a, z[0][r], z[kParts - 1][r]) : z[0][r];
      const int col = n0 + 16 * m + 4 * g;
      bf16_t* out = reinterpret_cast<bf16_t*>(a.out) + (int64_t)pair * a.out_stride + col;
      if (r0 + i16 < rows && col < (kGlu ? a.N / 2 : a.N)) *reinterpret_cast<uint2*>(out) = make_uint2(pack2<bf16_t>(o[0], o[1]), pack2<bf16_t>(o[2], o[3]));
    }
    __syncthreads();
  }
}

// any: workgroup = (16 outputs, expert, every gridDim.z-th 16 sorted rows), one dot product (two with the gate) per thread.
template <typename T, int kGlu>
__global__ __launch_bounds__(256) void moe_linear_any_kernel(const ExpertLinearArgs a) {
  constexpr int kStep = 64, NT = kGlu ? 2 : 1;
  __shared__ float xs[16][kStep + 1], ws[NT][16][kStep + 1];
  const int tid = threadIdx.x, r = tid >> 4, c = tid & 15, e = blockIdx.y, n0 = blockIdx.x * 16;
  const int first = a.row_start[e], last = a.row_start[e + 1];
  for (int base = first + 16 * blockIdx.z; base < last; base += 16 * gridDim.z) {
    float acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n] = 0.f;
    for (int k0 = 0; k0 < a.K; k0 += kStep) {
      for (int i = tid; i < 16 * kStep; i += 256) {
        const int rr = i / kStep, k = k0 + i % kStep, at = base + rr;
        float xv = 0.f;
        if (at < last && k < a.K)
          xv = to_float(reinterpret_cast<const T*>(a.x)[(int64_t)(a.per_token ? a.sorted_pair[at] / a.per_token : at) * a.x_stride + k]);
        xs[rr][i % kStep] = xv;
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const int wr = kGlu ? ((n0 + rr) >> 5) * 64 + ((n0 + rr) & 31) + 32 * n : n0 + rr;
          ws[n][rr][i % kStep] = wr < a.N && k < a.K ? to_float(reinterpret_cast<const T*>(a.w)[((int64_t)e * a.N + wr) * a.K + k]) : 0.f;
        }
      }
      __syncthreads();
#pragma unroll 16
      for (int k = 0; k < kStep; ++k)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = fmaf(xs[r][k], ws[n][c][k], acc[n]);
      __syncthreads();
    }
    if (base + r < last) {
      float o = acc[0];
      if constexpr (kGlu == kSiluGlu) o = acc[0] / (1.0f + expf(-acc[0])) * acc[NT - 1];
      if constexpr (kGlu == kClampedGlu) {
        const float z = fminf(acc[0], a.limit);
        o = z / (1.0f + expf(-a.alpha * z)) * (fminf(fmaxf(acc[NT - 1], -a.limit), a.limit) + a.shift);
      }
      reinterpret_cast<T*>(a.out)[(int64_t)(base + r) * a.out_stride + n0 + c] = from_float<T>(o);
    }
  }
}

// The tile of rows and of weights that a workgroup of the tiled products takes; false: none.  Each XCD has an eighth of the (row tile,
// weight tile) pairs, to one: shares of whole row tiles left the last XCD a third of the others' work (66 tiles: seven of 9, one of 3).
// A share's pairs go by row tiles, in fours: workgroups of a four with the same weight tile follow one another, and where shares are
// whole row tiles, as with few experts, none of them is read by two XCDs.  Large tiles with few rows come behind all others (see kApartRows), shared evenly too: the chip's last round is made of
// short ones.  600 rows, top 6 of 64 with uneven routing, width 2048: 132 + 71 -> 101 + 62 us.
__device__ __forceinline__ bool find_tile(const ExpertLinearArgs& a, int block, int& tile, int& n_tile) {
  const int xcd = block & 7, j = block >> 3, n = a.n_tiles;
  const int whole = a.num_tiles[0], rest = a.num_tiles[1], per = (whole * n + 7) / 8;
  if (j >= per) {
    const int rest_per = (rest * n + 7) / 8, at = xcd * rest_per + j - per;
    tile = whole + at / n;
    n_tile = at % n;
    return j - per < rest_per && at < rest * n;
  }
  const int low = xcd * per, high = min(low + per, whole * n);
  if (low + j >= high) return false;
  pair_at(n, low, high, j, tile, n_tile);
  return true;
}

// Step of K that a workgroup starts with; it comes round to the ones before it at its end.  Rows a multiple of 4 KB long start in the same channel
// of the L2 and of the memory, and workgroups that walk K in step read the same place of all rows at a time: a few channels serve
// everybody.  Four groups of experts start a quarter of K apart and the weight tiles of an expert a step apart: x stays shared, and the
// order of a sum depends on expert and column alone.  us from the first step on and so: 300 rows, top 6 of 64 experts of 1536 x 2048 84 / 68, 600
// rows 115 / 94, 8192 rows 354 / 336; of 2560 x 4096, 8192 rows 1390 / 1345, 32 rows 211 / 209.  Other rows (K of 768 and 1280): no difference.
__device__ __forceinline__ int first_step(int K, int e, int n_tile, int steps) {
  return K % 2048 == 0 ? ((e & 3) * (steps >> 2) + n_tile) % steps : 0;
}

// many: 128 weight rows x 32 kRows sorted rows per workgroup, four waves on v_mfma_f32_32x32x16_bf16.  Weights are the row
// operand and x the column operand, so that a lane ends with runs of four outputs of one row.  Steps of 64 along K through a
// ring of buffers in LDS that copies of later steps fill during this one; a row's eight 16-byte chunks trade places by half
// the row's number.  Consecutive workgroups of an XCD go through four row tiles for every weight tile.
// kRows 4: a wave has 64 x 64, two buffers.  kRows 2, where experts have so few rows that the stream of weights is the bound: a
// wave has 64 x 32, the small tile leaves LDS for three buffers of two workgroups per CU (72 KB of copies in flight or use each),
// and weights, read once by one workgroup, pass the caches by (nt).  900 pairs, 64 experts of 1536 x 2048 and 2048 x 768,
// weights from memory: 95 + 41 us as 128 x 128 tiles, 72 + 35 us (5.6 and 5.8 TB/s) as these; without nt 80 + 40, six buffers of one
// workgroup 70 + 41 (all before first_step).
template <int kGlu, int kRows>
__global__ __launch_bounds__(256, 2) void moe_linear_many_kernel(const ExpertLinearArgs a) {
  constexpr int kStages = kRows == 4 ? 2 : 3, kTile = 128, kK = 64;
  constexpr int kW = kTile * kK * 2, kStage = kW + 32 * kRows * kK * 2;   // bytes of the weights' part of a step, of a step
  constexpr int kM = kRows / 2, kCopies = 4 + kRows;       // 32-row blocks per wave; copies per thread and step
  __shared__ __attribute__((aligned(16))) char lds[kStages * kStage];     // [buffer][weights, x]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, hi = lane >> 5;
  // ---- which tile ----
  int n_tile, e, row0, row_end;
  const bool shared = kGlu != kClampedGlu && (int)blockIdx.x < a.shared.blocks;
  if (shared) {                                     // an XCD has all row tiles of some weight tiles: they are read once
    const int at = (int)(blockIdx.x & 7) * (a.shared.blocks >> 3) + (int)(blockIdx.x >> 3);
    n_tile = at / a.shared.row_tiles;
    if (n_tile >= a.shared.n_tiles) return;
    e = 0;
    row0 = at % a.shared.row_tiles * (32 * kRows);
    row_end = min(row0 + 32 * kRows, a.shared.rows);
  } else {
    int tile;
    if (!find_tile(a, (int)blockIdx.x - a.shared.blocks, tile, n_tile)) return;
    e = a.tile_expert[tile];
    row0 = a.tile_row[tile];
    row_end = min(row0 + 32 * kRows, a.row_start[e + 1]);
  }
  const int n0 = n_tile * kTile, N = shared ? a.shared.N : a.N, K = shared ? a.shared.K : a.K;

  // ---- copies: chunks of either operand per thread and step ----
  const v4i w_rows = make_rsrc(shared ? reinterpret_cast<const char*>(a.shared.w) : reinterpret_cast<const char*>(a.w) + (int64_t)e * N * K * 2,
                               (uint32_t)((int64_t)N * K * 2));
  const v4i x_rows = make_rsrc(shared ? reinterpret_cast<const char*>(a.shared.x) : reinterpret_cast<const char*>(a.x), shared ? a.shared.x_bytes : a.x_bytes);
  const uint32_t x_stride = shared ? (uint32_t)a.shared.x_stride : (uint32_t)a.x_stride;
  uint32_t from_w[4], from_x[kRows];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = 256 * i + tid, r = c >> 3, p = (c & 7) ^ ((r >> 1) & 7);
    const int row = min(n0 + r, N - 1);
    from_w[i] = (uint32_t)((shared ? shared_row<kGlu>(a, row) : row) * K + 8 * p) * 2u;
  }
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    const int c = 256 * i + tid, r = c >> 3, p = (c & 7) ^ ((r >> 1) & 7);
    const int at = min(row0 + r, row_end - 1);
    const uint32_t xr = (uint32_t)(a.per_token && !shared ? a.sorted_pair[at] / a.per_token : at);
    from_x[i] = (xr * x_stride + 8u * p) * 2u;
  }
  const int steps = K / kK, turn = first_step(K, e, n_tile, steps);
  const uint32_t lds_wave = lds_address(lds) + 1024 * wave;
  auto copy = [&](int step, int buffer) __attribute__((always_inline)) {      // past the last step nothing is read, and the count stays
    v4i w = w_rows, x = x_rows;
    if (kStages > 2) {
      w[2] = step < steps ? w[2] : 0;
      x[2] = step < steps ? x[2] : 0;
    }
    const uint32_t at = (uint32_t)(step < steps - turn ? step + turn : step + turn - steps) * (2 * kK), base = lds_wave + buffer * kStage;
    static_for<4>([&](auto I) { dma16_to_lds_at<4096 * decltype(I)::value, kRows == 2>(w, from_w[decltype(I)::value], at, base); });
    static_for<kRows>([&](auto I) { dma16_to_lds_at<kW + 4096 * decltype(I)::value>(x, from_x[decltype(I)::value], at, base); });
  };
  const int wn = wave & 1, wm = wave >> 1;          // the wave's half of the weight rows and of the rows
  // places of this lane's fragments: row l32 of a 32-row block, chunk 2 st + hi
  const int sw = (l32 >> 1) & 7;
  const char* frag = lds + l32 * 128;
  v16f acc[2][kM];
#pragma unroll
  for (int n = 0; n < 2; ++n)
#pragma unroll
    for (int m = 0; m < kM; ++m)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[n][m][r] = 0.f;

  static_for<kStages - 1>([&](auto I) { copy(decltype(I)::value, decltype(I)::value); });
  int buffer = 0;
  for (int step = 0; step < steps; ++step) {
    dma_wait_but<kCopies * (kStages - 2)>();
    workgroup_barrier();                            // this step's operands are there, the buffer of the step before is free
    if (kStages > 2 || step + 1 < steps) copy(step + kStages - 1, buffer == 0 ? kStages - 1 : buffer - 1);
    const char* wb = frag + buffer * kStage + wn * 64 * 128;
    const char* xb = frag + buffer * kStage + kW + wm * (32 * kM) * 128;
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      const int p = ((2 * st + hi) ^ sw) << 4;
      uint4 wf[2], xf[kM];
#pragma unroll
      for (int i = 0; i < 2; ++i) wf[i] = *reinterpret_cast<const uint4*>(wb + i * 32 * 128 + p);
#pragma unroll
      for (int i = 0; i < kM; ++i) xf[i] = *reinterpret_cast<const uint4*>(xb + i * 32 * 128 + p);
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int m = 0; m < kM; ++m) acc[n][m] = mfma32x32x16<bf16_t>(wf[n], xf[m], acc[n][m]);
    }
    buffer = buffer + 1 == kStages ? 0 : buffer + 1;
  }
  if (kStages > 2) dma_wait_all();                  // (copies past the last step)
  // ---- lane: row l32 of a block, weight rows 8 (r / 4) + 4 hi + r % 4 ----
  bf16_t* const out_of = shared ? a.shared.out : reinterpret_cast<bf16_t*>(a.out);
  const int64_t out_stride = shared ? a.shared.out_stride : a.out_stride;
#pragma unroll
  for (int m = 0; m < kM; ++m) {
    const int row = row0 + (wm * kM + m) * 32 + l32;
    if (row >= row_end) continue;
    bf16_t* out = out_of + (int64_t)row * out_stride;
#pragma unroll
    for (int r = 0; r < 16; r += 4) {
      if constexpr (kGlu) {
        const int col = (n0 + wn * 64) / 2 + 2 * r + 4 * hi;
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = glu_of<kGlu>(a, acc[0][m][r + i], acc[1][m][r + i]);
        if (2 * col < N) *reinterpret_cast<uint2*>(out + col) = make_uint2(pack2<bf16_t>(o[0], o[1]), pack2<bf16_t>(o[2], o[3]));
      } else {
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          const int col = n0 + wn * 64 + 32 * n + 2 * r + 4 * hi;
          if (col < N)
            *reinterpret_cast<uint2*>(out + col) = make_uint2(pack2<bf16_t>(acc[n][m][r], acc[n][m][r + 1]),
                                                              pack2<bf16_t>(acc[n][m][r + 2], acc[n][m][r + 3]));
        }
      }
    }
  }
}

// many, few workgroups: 64 weight rows x 32 kBlocks sorted rows per workgroup, whose waves take a sixteen of K each of every step and add up in LDS, in 32 bits.
// Weights are the bound as in the 64-row form above, but where that has fewer workgroups than CUs, each of them waits for its own three buffers: 16 KB
// of weights in flight per CU.  Half as many weight rows are twice as many workgroups, and six buffers (five with 64 rows) 40 KB (32) in flight for each of
// two per CU.  narrow_pays has when.  us of a product, 64-row form / this: 6 pairs, 64 experts of 1536 x 2048 with the gate 17.5 / 10.2 and of
// 2048 x 768 9.2 / 7.1; 4 pairs of 2560 x 4096 31.3 / 18.0 (4.7 TB/s), 12 of 4096 x 1280 24.8 / 20.9; one of 4096 x 14336 92.9 / 43.1.
template <int kGlu, int kBlocks>
__global__ __launch_bounds__(256, 2) void moe_linear_narrow_kernel(const ExpertLinearArgs a) {
  constexpr int kStages = kBlocks == 1 ? 6 : 5, kTile = 64, kRows = 32 * kBlocks, kK = 64, kW = kTile * kK * 2, kStage = kW + kRows * kK * 2, kCopies = 2 + kBlocks;
  __shared__ __attribute__((aligned(16))) char lds[kStages * kStage];     // [buffer][weights, x]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, hi = lane >> 5;
  // ---- which tile ----
  int n_tile, e, row0, row_end;
  const bool shared = kGlu != kClampedGlu && (int)blockIdx.x < a.shared.blocks;
  if (shared) {
    const int at = (int)(blockIdx.x & 7) * (a.shared.blocks >> 3) + (int)(blockIdx.x >> 3);
    n_tile = at / a.shared.row_tiles;
    if (n_tile >= a.shared.n_tiles) return;
    e = 0;
    row0 = at % a.shared.row_tiles * kRows;
    row_end = min(row0 + kRows, a.shared.rows);
  } else {
    int tile;
    if (!find_tile(a, (int)blockIdx.x - a.shared.blocks, tile, n_tile)) return;
    e = a.tile_expert[tile];
    row0 = a.tile_row[tile];
    row_end = min(row0 + kRows, a.row_start[e + 1]);
  }
  const int n0 = n_tile * kTile, N = shared ? a.shared.N : a.N, K = shared ? a.shared.K : a.K;

  // ---- copies: two chunks of weights and kBlocks of x per thread and step ----
  const v4i w_rows = make_rsrc(shared ? reinterpret_cast<const char*>(a.shared.w) : reinterpret_cast<const char*>(a.w) + (int64_t)e * N * K * 2,
                               (uint32_t)((int64_t)N * K * 2));
  const v4i x_rows = make_rsrc(shared ? reinterpret_cast<const char*>(a.shared.x) : reinterpret_cast<const char*>(a.x), shared ? a.shared.x_bytes : a.x_bytes);
  const int r0 = tid >> 3, p0 = (tid & 7) ^ ((r0 >> 1) & 7);       // (row r0 + 32 has the same swizzle)
  uint32_t from_w[2], from_x[kBlocks];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = min(n0 + r0 + 32 * i, N - 1);
    from_w[i] = (uint32_t)((shared ? shared_row<kGlu>(a, row) : row) * K + 8 * p0) * 2u;
  }
#pragma unroll
  for (int i = 0; i < kBlocks; ++i) {
    const int at = min(row0 + r0 + 32 * i, row_end - 1);
    const uint32_t xr = (uint32_t)(a.per_token && !shared ? a.sorted_pair[at] / a.per_token : at);
    from_x[i] = (xr * (shared ? (uint32_t)a.shared.x_stride : (uint32_t)a.x_stride) + 8u * p0) * 2u;
  }
  const int steps = K / kK, turn = first_step(K, e, n_tile, steps);
  const uint32_t lds_wave = lds_address(lds) + 1024 * wave;
  auto copy = [&](int step, int buffer) __attribute__((always_inline)) {      // past the last step nothing is read, and the count stays
    v4i w = w_rows, x = x_rows;
    w[2] = step < steps ? w[2] : 0;
    x[2] = step < steps ? x[2] : 0;
    const uint32_t at = (uint32_t)(step < steps - turn ? step + turn : step + turn - steps) * (2 * kK), base = lds_wave + buffer * kStage;
    dma16_to_lds_at<0, true>(w, from_w[0], at, base);
    dma16_to_lds_at<4096, true>(w, from_w[1], at, base);
    static_for<kBlocks>([&](auto I) { dma16_to_lds_at<kW + 4096 * decltype(I)::value>(x, from_x[decltype(I)::value], at, base); });
  };
  // this lane's fragments of the wave's sixteen: row l32 of a 32-row block, chunk 2 wave + hi
  const char* frag = lds + l32 * 128 + (((2 * wave + hi) ^ ((l32 >> 1) & 7)) << 4);
  v16f acc[kBlocks][2];
#pragma unroll
  for (int m = 0; m < kBlocks; ++m)
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[m][n][r] = 0.f;

  static_for<kStages - 1>([&](auto I) { copy(decltype(I)::value, decltype(I)::value); });
  int buffer = 0;
  for (int step = 0; step < steps; ++step) {
    dma_wait_but<kCopies * (kStages - 2)>();
    workgroup_barrier();                            // this step's operands are there, the buffer of the step before is free
    copy(step + kStages - 1, buffer == 0 ? kStages - 1 : buffer - 1);
    const char* at = frag + buffer * kStage;
    const uint4 w0 = *reinterpret_cast<const uint4*>(at), w1 = *reinterpret_cast<const uint4*>(at + 32 * 128);
    uint4 x[kBlocks];
#pragma unroll
    for (int m = 0; m < kBlocks; ++m) x[m] = *reinterpret_cast<const uint4*>(at + kW + m * 32 * 128);
#pragma unroll
    for (int m = 0; m < kBlocks; ++m) {
      acc[m][0] = mfma32x32x16<bf16_t>(w0, x[m], acc[m][0]);
      acc[m][1] = mfma32x32x16<bf16_t>(w1, x[m], acc[m][1]);
    }
    buffer = buffer + 1 == kStages ? 0 : buffer + 1;
  }
  dma_wait_all();                                   // (copies past the last step)
  __syncthreads();
  // ---- the waves' sums: 16-byte pieces [wave][block of outputs][four of a lane][lane]; wave w finishes the w-th four of every block.  Lane: row l32,
  // weight rows 8 w + 4 hi + 0 .. 3 ----
  static_assert(4 * 2 * kBlocks * 4 * 64 * 16 <= kStages * kStage, "the sums' room");
  float4* const sums = reinterpret_cast<float4*>(lds);
#pragma unroll
  for (int m = 0; m < kBlocks; ++m)
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        sums[(((wave * kBlocks + m) * 2 + n) * 4 + i) * 64 + lane] = make_float4(acc[m][n][4 * i], acc[m][n][4 * i + 1], acc[m][n][4 * i + 2], acc[m][n][4 * i + 3]);
  __syncthreads();
  bf16_t* const out_of = shared ? a.shared.out : reinterpret_cast<bf16_t*>(a.out);
  const int64_t out_stride = shared ? a.shared.out_stride : a.out_stride;
  const int r = 8 * wave + 4 * hi;
#pragma unroll
  for (int m = 0; m < kBlocks; ++m) {
    const int row = row0 + 32 * m + l32;
    if (row >= row_end) continue;
    float v[2][4];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      float4 x[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) x[w] = sums[(((w * kBlocks + m) * 2 + n) * 4 + wave) * 64 + lane];
      v[n][0] = (x[0].x + x[1].x) + (x[2].x + x[3].x);
      v[n][1] = (x[0].y + x[1].y) + (x[2].y + x[3].y);
      v[n][2] = (x[0].z + x[1].z) + (x[2].z + x[3].z);
      v[n][3] = (x[0].w + x[1].w) + (x[2].w + x[3].w);
    }
    bf16_t* out = out_of + (int64_t)row * out_stride;
    if constexpr (kGlu) {
      float o[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = glu_of<kGlu>(a, v[0][i], v[1][i]);
      *reinterpret_cast<uint2*>(out + n0 / 2 + r) = make_uint2(pack2<bf16_t>(o[0], o[1]), pack2<bf16_t>(o[2], o[3]));
    } else {
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const int col = n0 + 32 * n + r;
        if (col < N) *reinterpret_cast<uint2*>(out + col) = make_uint2(pack2<bf16_t>(v[n][0], v[n][1]), pack2<bf16_t>(v[n][2], v[n][3]));
      }
    }
  }
}

// many, large tiles: 256 sorted rows x 256 weight rows, four waves of 128 x 128 (a wave's accumulators fill half its SIMD's
// registers; per flop it reads half as much of LDS as with 64 x 64).  The operands of a 16-wide step are read during the
// products of the one before; a step's last products hide the barrier, after which the next step's operands are there and
// more copies start: x, which other workgroups of the XCD read too, one step ahead in two buffers, the weights, which come
// from memory, two steps ahead in three.  Together they fill the LDS.  What x waits for bounds a step: its copies right behind a barrier that is as early as
// the last reads allow (4096 wide, random numbers, 8 rounds of tiles: 1176 TFLOP/s with the barrier at the fourth product and copies from the eighth, 1235
// from the fourth, 1276 so; a barrier in the sixteen before for the copies and one for the reads: 1272).  Then comes power: the same product of zeros 1340 to 1670.
// A workgroup stays on its CU and takes every a.groups-th tile of its XCD, because the way into a tile was as long as six to eight steps of K: its number,
// expert and rows (one load for the other, 5 us under load), the first copies (3.5), and behind the steps the stores (4.5).  The tile behind is
// known and its rows' places are loaded a tile ahead, its first copies run beside the stores, and these go through LDS, since a lane's runs of eight outputs
// in 32 rows took the address unit four times as long as whole rows do.  us: 65536 rows, 2048 x 768 268 -> 229, 2048 x 2048 498 -> 472; both
// products of 8192 rows, top 6 of 64, routed unevenly, 1536 x 2048 with the gate 359 -> 337, 2048 x 768 238 -> 219.
// With K of 4096 and more and two and a half rounds, the way into a tile is little of it and uneven tiles are more: there every tile has a workgroup of its
// own again and goes where a CU is free.  us, 64 experts of 2560 x 4096 with the gate, 60 / 160 / 200 / 300 rows each, strided 294 / 366 / 381 / 500, so 278 / 342 /
// 378 / 475, of 3072 x 4096 340 / 449 / 499 / 617 and 335 / 433 / 495 / 601 (a round and a quarter, 32 experts of 2560 x 4096, 80 rows 159 and 166).
// Halves: tiles of the last round in halves gain a quarter of a tile (64 experts of 1536 x 2048 with the gate, 132 rows each 113 / 104 without / with), but where
// tiles of few rows were to fill that round they come one round later: 156 rows 116 / 126, 180 120 / 131.
// (Halves that have no rows, of tiles of at most 128, are run all the same: without them 108 sizes took 0.98 to 1.07 of the time, 1.008 on average.)
template <int kGlu>
__global__ __launch_bounds__(256, 1) void moe_linear_large_kernel(const ExpertLinearArgs a) {
  constexpr int kTile = 256, kK = 64, kStage = kTile * kK * 2;       // bytes of one operand's step
  __shared__ __attribute__((aligned(16))) char lds[5 * kStage];      // weights three times, x twice
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, hi = lane >> 5;
  // ---- this workgroup's tiles: every a.groups-th of its XCD's ----
  const LargeShare share(a.n_tiles, a.num_tiles[0], a.num_tiles[1], kGlu == kClampedGlu ? 0 : a.shared.row_tiles, a.shared.n_tiles, a.shared.units,
                         blockIdx.x & 7, a.groups);
  struct Tile { int e, row0, rows, n_tile; };           // (e: a.experts for the shared one)
  auto find = [&](int j, Tile& t) __attribute__((always_inline)) {
    TilePlace place;
    if (!share.find(j, place)) return false;
    t.n_tile = place.n_tile;
    t.rows = place.half < 0 ? kTile : kTile / 2;
    if (place.shared) {
      t.e = a.experts;
      t.row0 = place.tile * kTile;
    } else {
      t.e = a.tile_expert[place.tile];
      t.row0 = a.tile_row[place.tile] + (place.half > 0 ? kTile / 2 : 0);
    }
    return true;
  };
  auto is_shared = [&](const Tile& t) __attribute__((always_inline)) { return kGlu != kClampedGlu && t.e == a.experts; };
  auto after_it = [&](const Tile& t) __attribute__((always_inline)) { return a.groups * (is_shared(t) ? a.shared.units : 1); };
  auto end_of = [&](const Tile& t) __attribute__((always_inline)) { return min(t.row0 + t.rows, is_shared(t) ? a.shared.rows : a.row_start[t.e + 1]); };
  int j = blockIdx.x >> 3;
  Tile now{}, next{};
  if (!find(j, now)) return;
  j += after_it(now);
  bool more = find(j, next);

  const int total = a.row_start[a.experts];
  // the rows of x that this thread copies: those of the sorted rows row0 + (256 i + tid) / 8.  Past the tile's end they are the next
  // expert's, whose results are not stored.
  auto pairs_of = [&](const Tile& t, uint32_t (&pair)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int at = min(t.row0 + ((256 * i + tid) >> 3), (is_shared(t) ? a.shared.rows : total) - 1);
      pair[i] = (uint32_t)(a.per_token && !is_shared(t) ? a.sorted_pair[at] : at);
    }
  };
  uint32_t from_w[8], from_x[8], pair[8];
  v4i w_rows, x_rows;
  int steps, turn;
  auto places_of = [&](const Tile& t) __attribute__((always_inline)) {
    const bool shared = is_shared(t);
    const int N = shared ? a.shared.N : a.N, K = shared ? a.shared.K : a.K;
    w_rows = make_rsrc(shared ? reinterpret_cast<const char*>(a.shared.w) : reinterpret_cast<const char*>(a.w) + (int64_t)t.e * N * K * 2,
                       (uint32_t)((int64_t)N * K * 2));
    x_rows = make_rsrc(shared ? reinterpret_cast<const char*>(a.shared.x) : reinterpret_cast<const char*>(a.x), shared ? a.shared.x_bytes : a.x_bytes);
    const uint32_t x_stride = shared ? (uint32_t)a.shared.x_stride : (uint32_t)a.x_stride;
    steps = K / kK;
    turn = first_step(K, t.e, t.n_tile, steps);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int c = 256 * i + tid, r = c >> 3, p = (c & 7) ^ ((r >> 1) & 7);
      const int w_row = min(t.n_tile * kTile + r, N - 1);
      from_w[i] = (uint32_t)((shared ? shared_row<kGlu>(a, w_row) : w_row) * K + 8 * p) * 2u;
      uint32_t row = pair[i];
      if (a.per_token && !shared) {                            // pair / per_token: the quotient of the rounded factor is that or one less
        row = __umulhi(pair[i], a.token_factor);
        row += pair[i] - row * (uint32_t)a.per_token >= (uint32_t)a.per_token;
      }
      from_x[i] = (row * x_stride + 8u * p) * 2u;
    }
  };
  constexpr int kX = 3 * kStage;                    // where x begins
  const uint32_t lds_wave = lds_address(lds) + 1024 * wave;
  auto k_of = [&](int step) __attribute__((always_inline)) { return (uint32_t)(step < steps - turn ? step + turn : step + turn - steps) * (2 * kK); };
  // copy i of eight of a step's operand; past the last step nothing is read (the buffer is not used again)
  auto copy_w = [&](auto I, int step, uint32_t buffer) __attribute__((always_inline)) {
    v4i rows = w_rows;
    rows[2] = step < steps ? rows[2] : 0;
    dma16_to_lds_at<4096 * decltype(I)::value>(rows, from_w[decltype(I)::value], k_of(step), lds_wave + buffer);
  };
  auto copy_x = [&](auto I, int step) __attribute__((always_inline)) {
    v4i rows = x_rows;
    rows[2] = step < steps ? rows[2] : 0;
    dma16_to_lds_at<4096 * decltype(I)::value>(rows, from_x[decltype(I)::value], k_of(step), lds_wave + kX + (step & 1) * kStage);
  };
  auto copy_first = [&](int blocks) __attribute__((always_inline)) {       // the first step's operands, then the second's weights
    static_for<8>([&](auto I) { copy_w(I, 0, 0); });
    static_for<8>([&](auto I) {
      if (decltype(I)::value < 2 * blocks) copy_x(I, 0);
    });
    static_for<8>([&](auto I) { copy_w(I, 1, kStage); });
  };
  const int wn = wave & 1, wm = wave >> 1;
  const int sw = (l32 >> 1) & 7;
  const char* frag = lds + l32 * 128;
  v16f acc[4][4];
  uint4 wf[2][4], xf[2][4];
  // where this lane's operands of the four 16-wide steps lie in a buffer
  uint32_t place[4];
#pragma unroll
  for (int st = 0; st < 4; ++st) place[st] = ((2 * st + hi) ^ sw) << 4;
  const char* w_frag = frag + wn * (128 * 128);
  const char* x_frag = frag + wm * (32 * 128) + kX;
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};
  // The product with kBlocks blocks of 32 rows for each wave, those of the two halves in turns: a tile that is not whole takes no more
  // time than its rows do.
  auto run = [&](auto BLOCKS) __attribute__((always_inline)) {
    constexpr int kBlocks = decltype(BLOCKS)::value, kProducts = 4 * kBlocks, kPer = kBlocks == 1 ? 2 : 1;
    constexpr int kBarrier = kBlocks == 4 ? 1 : kBlocks - 1;         // the product of the last sixteen with the step's barrier, before the next step's reads
    // The products of a 16-wide step one by one; after each of them one of the next step's reads (every kEvery-th from product
    // kFirst on, those that are needed first come first) and whatever `also` does: the matrix unit must not wait for a queue of
    // reads or copies.
    auto products = [&](auto SET, auto FIRST, auto EVERY, const char* wb, const char* xb, auto&& also) __attribute__((always_inline)) {
      constexpr int set = decltype(SET)::value, next = set ^ 1, kFirst = decltype(FIRST)::value, kEvery = decltype(EVERY)::value;
      static_for<kProducts>([&](auto I) {
        constexpr int i = decltype(I)::value, n = i / kBlocks, m = i % kBlocks;
        acc[n][m] = mfma32x32x16<bf16_t>(wf[set][n], xf[set][m], acc[n][m]);
        also(I);
        if constexpr (i >= kFirst && (i - kFirst) % kEvery == 0) {
          static_for<kPer>([&](auto Q) {
            constexpr int j = (i - kFirst) / kEvery * kPer + decltype(Q)::value;
            if constexpr (j >= 1 && j <= kBlocks) xf[next][j - 1] = *reinterpret_cast<const uint4*>(xb + (j - 1) * 64 * 128);
            else if constexpr (j < 4 + kBlocks) {
              constexpr int w = j == 0 ? 0 : j - kBlocks;
              wf[next][w] = *reinterpret_cast<const uint4*>(wb + w * 32 * 128);
            }
          });
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    constexpr std::integral_constant<int, kBlocks == 4 ? 2 : 1> spread{};
    auto nothing = [](auto) {};

    dma_wait_all();                                 // the first copies; what the tile before stored
    __syncthreads();
    static_for<2 * kBlocks>([&](auto I) { copy_x(I, 1); });
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      wf[0][i] = *reinterpret_cast<const uint4*>(w_frag + place[0] + i * 32 * 128);
      if (i < kBlocks) xf[0][i] = *reinterpret_cast<const uint4*>(x_frag + place[0] + i * 64 * 128);
    }
    uint32_t w_at = 0;                              // the weights' buffer of this step, in bytes
    for (int step = 0; step < steps; ++step) {
      const uint32_t w_next = w_at == 2 * kStage ? 0 : w_at + kStage, w_free = w_at == 0 ? 2 * kStage : w_at - kStage;
      const char* wb = w_frag + w_at;
      const char* xb = x_frag + (step & 1) * kStage;
      // the weights two steps ahead, into the buffer that the step before this one has left
      products(c0, c1, spread, wb + place[1], xb + place[1], [&](auto I) {
        constexpr int i = decltype(I)::value;
        if constexpr (kBlocks == 4) {
          if constexpr (i % 2 == 0) copy_w(std::integral_constant<int, i / 2>{}, step + 2, w_free);
        } else if constexpr (i * kPer < 8)
          static_for<kPer>([&](auto Q) { copy_w(std::integral_constant<int, i * kPer + decltype(Q)::value>{}, step + 2, w_free); });
      });
      products(c1, c1, spread, wb + place[2], xb + place[2], nothing);
      products(c0, c1, spread, wb + place[3], xb + place[3], nothing);
      // the next step's operands have to be there before its first reads, and this step's have been read: then x two steps
      // ahead follows into its buffer.  What may be in flight until then are the eight copies of weights from above.
      products(c1, BLOCKS, c1, w_frag + w_next + place[0], x_frag + ((step & 1) ^ 1) * kStage + place[0], [&](auto I) {
        constexpr int i = decltype(I)::value;
        if constexpr (i == kBarrier) {
          dma_wait_but<8>();
          workgroup_barrier();
        }
        if constexpr (i > kBarrier && i <= kBarrier + 2 * kBlocks) copy_x(std::integral_constant<int, i - kBarrier - 1>{}, step + 2);
      });
      w_at = w_next;
    }
    dma_wait_all();                                 // (copies past the last step)
  };
  pairs_of(now, pair);
  places_of(now);
  // (a second half without rows is one block whose results are not stored)
  int row_end = end_of(now), blocks = max((row_end - now.row0 + 63) / 64, 1);
  copy_first(blocks);
  for (;;) {
    int next_end = 0;
    Tile after{};
    bool and_more = false;
    if (more) {                                     // what the boundary behind this tile needs, here already
      pairs_of(next, pair);
      next_end = end_of(next);
      j += after_it(next);
      and_more = find(j, after);
    }
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[n][m][r] = 0.f;
    switch (blocks) {
      case 1: run(c1); break;
      case 2: run(std::integral_constant<int, 2>{}); break;
      case 3: run(std::integral_constant<int, 3>{}); break;
      default: run(std::integral_constant<int, 4>{});
    }
    workgroup_barrier();                            // the last step's operands have been read
    const Tile of = now;
    const int end = row_end;
    if (more) {
      now = next;
      next = after;
      row_end = next_end;
      blocks = max((row_end - now.row0 + 63) / 64, 1);
      places_of(now);
      copy_first(blocks);
    }
    // ---- lane: row l32 of a block, weight rows 8 (r / 4) + 4 hi + r % 4; halves of the wave trade runs of four, so that a lane has eight outputs
    // in a row, and a block's rows go through LDS, the wave's 8 KB of the third weights' or of the second x buffer, which the next tile's first copies
    // leave alone, so that a store's lanes are whole rows ----
    constexpr int kChunks = kGlu ? 8 : 16, kRowsPer = 64 / kChunks;        // 16-byte chunks of a wave's output row; rows of a store
    auto place_of = [&](int row, int chunk) __attribute__((always_inline)) {
      return row * (16 * kChunks) + ((chunk ^ ((kGlu ? row >> 1 : row) & (kChunks - 1))) << 4);
    };
    const bool of_shared = is_shared(of);
    bf16_t* const out_of = of_shared ? a.shared.out : reinterpret_cast<bf16_t*>(a.out);
    const int64_t out_stride = of_shared ? a.shared.out_stride : a.out_stride;
    const int of_N = of_shared ? a.shared.N : a.N, out_cols = kGlu ? of_N / 2 : of_N, col0 = (of.n_tile * kTile + wn * 128) / (kGlu ? 2 : 1);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      if (of.row0 + 32 * (wm + 2 * m) >= end) break;
      char* const own = lds + (m & 1 ? 4 : 2) * kStage + 8192 * wave;
      if constexpr (kGlu != kNoGlu) {                // a block's sums leave their registers only now
#pragma unroll
        for (int n = 0; n < 4; ++n) asm volatile("" : "+a"(acc[n][m]));
      }
#pragma unroll
      for (int n = 0; n < (kGlu ? 2 : 4); ++n) {
#pragma unroll
        for (int r = 0; r < 16; r += 8) {
          float o[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            if constexpr (kGlu) o[i] = glu_of<kGlu>(a, acc[2 * n][m][r + i], acc[2 * n + 1][m][r + i]);
            else o[i] = acc[n][m][r + i];
          }
          const auto x = __builtin_amdgcn_permlane32_swap(pack2<bf16_t>(o[0], o[1]), pack2<bf16_t>(o[4], o[5]), false, false);
          const auto y = __builtin_amdgcn_permlane32_swap(pack2<bf16_t>(o[2], o[3]), pack2<bf16_t>(o[6], o[7]), false, false);
          *reinterpret_cast<uint4*>(own + place_of(l32, 4 * n + (r >> 2) + hi)) = make_uint4(x[0], y[0], x[1], y[1]);
        }
      }
      __builtin_amdgcn_wave_barrier();
      const int chunk = lane % kChunks, col = col0 + 8 * chunk;
      const int row = of.row0 + 32 * (wm + 2 * m) + lane / kChunks;
      bf16_t* out = out_of + (int64_t)row * out_stride + col;
#pragma unroll
      for (int i = 0; i < 32 / kRowsPer; ++i) {
        const uint4 v = *reinterpret_cast<const uint4*>(own + place_of(kRowsPer * i + lane / kChunks, chunk));
        if (row + kRowsPer * i < end && col < out_cols) *reinterpret_cast<uint4*>(out + (int64_t)(kRowsPer * i) * out_stride) = v;
      }
      __builtin_amdgcn_wave_barrier();
    }
    if (!more) break;
    more = and_more;
  }
}

// Rows of a tile: large ones where experts have enough rows on average to fill them, small ones where most experts fit in one.
static int tile_rows(int64_t pairs, int experts) {
  return pairs >= kLargeTileRows * (int64_t)experts ? 256 : pairs > kSmallTileRows * (int64_t)experts ? 128 : 64;
}
static int64_t max_tiles(int64_t pairs, int experts, int rows) { return (pairs + rows - 1) / rows + experts; }
// Whether a product's weights go in 64 rows per workgroup instead of 128, by the workgroups of 128 to be expected where routing is even.  Up to 160 these leave CUs
// idle: 1.03 to 2.2 times as fast at K of 768 to 14336 (1.27 and more up to 128 workgroups).  From 160 to 248 both fill the chip about once, 0.95 to 1.10.
// From 248 to 384 a part of the CUs has two of 128 and the others one, while all have two of 64: 1.03 to 1.19 (K 768: 1.05 up to 328, 0.93 at 396).  At 400 to 500
// 0.89 to 1.04, and above it 0.96 to 1.1 where there are many steps of K, 0.8 to 0.95 where there are few.  More than four pairs per expert were not faster (mixtures
// of 64 experts: 0.98 at six, 0.88 at 28).  With the gate it is 0.01 to 0.04 more, with the clamped one 0.01 to 0.08.  K of 512 to 704: 1.2
// to 1.45 up to 115 workgroups too, but 0.78 to 1.06 from 163 on (six buffers' start and the sums at the end are longer than eight to eleven steps): not taken.
static bool narrow_pays(int64_t pairs, int experts, int N, int K, const ExpertLinearArgs::Shared& shared) {
  const int least_k = shared.rows != 0 ? std::min(K, shared.K) : K;
  if (pairs > 4 * (int64_t)experts || least_k < 768) return false;
  const float with_rows = (float)experts * (1.f - powf(1.f - 1.f / (float)experts, (float)pairs));
  const float wgs = with_rows * (float)((N + 127) / 128) + (shared.rows != 0 ? (float)((shared.rows + 63) / 64) * (float)((shared.N + 127) / 128) : 0.f);
  return wgs <= 160.f || (wgs >= 248.f && wgs <= (least_k >= 1024 ? 384.f : 328.f));
}
// Tiles of 256 rows and weight rows to be expected.
static int64_t large_tiles(int64_t pairs, int experts, int N) {
  const int64_t rows = pairs / 256 + experts / 2;
  return (N + 255) / 256 * (rows > experts ? rows : experts);
}
// Whether a product of N outputs runs on the tiles of 256 rows of a plan that has both.  With 48 to 384 rows per expert a large tile has one to four of its
// blocks of 64 rows; it reads every weight once for the expert's rows and half as much of LDS per flop, but has a CU to itself: it pays where there is one
// for each CU and N fills it.  us as 128 and 256 rows, weights from memory, top 4 routed unevenly, 50 / 80 / 120 / 340 rows each: 64 experts of 1536 x 2048 with
// the gate (384 tiles and more) 98 99 125 208 / 94 101 105 168, of 2048 x 768 57 59 71 132 / 55 60 61 96, of 2560 x 4096 282 331 365 722 / 268 295 313 531; 32 of
// 2048 x 1024 (256 tiles) 42 44 48 87 / 36 50 50 62.  370 batches of 16 to 128 experts, 49 to 1500 rows each, from 256 tiles on: 0.944 of the time that the rule before took,
// 640 tiles or 384 of many rows; what loses has a few rows more than a block on average (70 to 115 rows; worst 32 of 3072 x 1024 with the gate, 76 rows 56 / 61,
// 64 of 1024 x 2048, 95 rows 86 / 90).  Below: 32 of 1536 x 2048 (192) 48 49 75 111 / 48 53 51 85, 16 of 1024 x 2048 (64 tiles), 56 rows 33 / 33.
static bool large_tiles_pay(int64_t pairs, int experts, int N) {
  if (8 * (256 * ((N + 255) / 256) - N) > N) return false;
  return large_tiles(pairs, experts, N) >= 256;
}
static int plan_blocks(int64_t pairs) { return (int)((pairs + kPlanPairs - 1) / kPlanPairs); }

}  // namespace mvllm

using namespace mvllm;

static int route(RouteArgs a, int64_t rows, void* stream) {
  if (rows < 0 || a.experts <= 0 || a.top <= 0 || a.top > a.experts || a.groups <= 0 || a.experts % a.groups != 0 || a.keep <= 0 ||
      a.keep > a.groups || a.z_stride < a.experts || (int64_t)a.keep * (a.experts / a.groups) < a.top || a.identity < 0 || a.identity > a.experts)
    return MVLLM_ERR_BAD_SHAPE;
  if (a.experts > kMaxExperts || a.top > 64 || a.groups > 64 || rows > (1 << 28)) return MVLLM_ERR_UNSUPPORTED;
  if (rows == 0) return MVLLM_OK;
  if (!a.ids || !a.weights || !a.z) return MVLLM_ERR_NULL_POINTER;
  a.rows = (int)rows;
  const dim3 grid((unsigned)((rows + 3) / 4)), block(256);
  hipStream_t s = (hipStream_t)stream;
  if (a.experts <= 64) moe_route_kernel<1><<<grid, block, 0, s>>>(a);
  else if (a.experts <= 128) moe_route_kernel<2><<<grid, block, 0, s>>>(a);
  else if (a.experts <= 256) moe_route_kernel<4><<<grid, block, 0, s>>>(a);
  else moe_route_kernel<16><<<grid, block, 0, s>>>(a);
  return launch_status();
}

extern "C" int mvllm_moe_route(int32_t* ids, float* weights, const float* logits, int64_t logit_row_stride,
                               const float* correction, int64_t rows, int experts, int top, int groups, int keep,
                               void* stream) {
  RouteArgs a = {};
  a.ids = ids; a.weights = weights; a.z = logits; a.correction = correction; a.z_stride = logit_row_stride;
  a.experts = experts; a.top = top; a.groups = groups; a.keep = keep; a.renormalize = true;
  return route(a, rows, stream);
}

extern "C" int mvllm_moe_route_softmax(int32_t* ids, float* weights, const float* logits, int64_t logit_row_stride,
                                       const float* correction, int64_t rows, int experts, int identity, int top,
                                       int renormalize, void* stream) {
  if (experts < 0 || identity < 0 || experts > kMaxExperts || identity > kMaxExperts) return MVLLM_ERR_BAD_SHAPE;
  RouteArgs a = {};
  a.ids = ids; a.weights = weights; a.z = logits; a.correction = correction; a.z_stride = logit_row_stride;
  a.experts = experts + identity; a.identity = identity; a.top = top; a.groups = 1; a.keep = 1; a.softmax = true;
  a.renormalize = renormalize != 0;
  return route(a, rows, stream);
}

extern "C" size_t mvllm_moe_plan_bytes(int64_t pairs, int experts) {
  if (pairs <= 0 || experts <= 0) return 0;
  const int rows = tile_rows(pairs, experts);
  const int64_t tiles = 2 * max_tiles(pairs, experts, rows) + 2 + (rows == 128 ? 2 * max_tiles(pairs, experts, 256) + 2 : 0);
  return (size_t)(2 * pairs + experts + 1 + tiles + (int64_t)plan_blocks(pairs) * experts + 4) * sizeof(int32_t);
}

// the parts of a plan, in order
static PlanArgs plan_parts_of(void* plan, const int32_t* ids, int64_t pairs, int experts) {
  PlanArgs a;
  a.ids = ids;
  a.place = reinterpret_cast<int32_t*>(plan);
  a.sorted_pair = a.place + pairs;
  a.row_start = a.sorted_pair + pairs;
  a.pairs = (int)pairs; a.experts = experts; a.blocks = plan_blocks(pairs);
  a.tile_rows = tile_rows(pairs, experts);
  int32_t* at = a.row_start + experts + 1;
  for (int i = 0; i < 2; ++i) {
    const int64_t most = i == 0 ? max_tiles(pairs, experts, a.tile_rows) : a.tile_rows == 128 ? max_tiles(pairs, experts, 256) : 0;
    a.tiles[i] = {at, at + most, at + 2 * most};
    at += most > 0 ? 2 * most + 2 : 0;
  }
  a.hist = at;
  return a;
}

extern "C" int mvllm_moe_plan(void* plan, size_t plan_bytes, const int32_t* ids, int64_t pairs, int experts, void* stream) {
  if (pairs < 0 || experts <= 0) return MVLLM_ERR_BAD_SHAPE;
  if (experts > kMaxExperts || pairs > (1 << 30)) return MVLLM_ERR_UNSUPPORTED;
  if (pairs == 0) return MVLLM_OK;
  if (!plan || !ids) return MVLLM_ERR_NULL_POINTER;
  if (plan_bytes < mvllm_moe_plan_bytes(pairs, experts)) return MVLLM_ERR_WORKSPACE;
  const PlanArgs a = plan_parts_of(plan, ids, pairs, experts);
  hipStream_t s = (hipStream_t)stream;
  if (a.blocks > 1) moe_count_kernel<<<dim3((unsigned)a.blocks), dim3(256), 0, s>>>(a);
  const dim3 grid((unsigned)a.blocks), block(1024);
  if (a.tile_rows == 64) moe_place_kernel<64><<<grid, block, 0, s>>>(a);
  else if (a.tile_rows == 128) moe_place_kernel<128><<<grid, block, 0, s>>>(a);
  else moe_place_kernel<256><<<grid, block, 0, s>>>(a);
  return launch_status();
}

// f(a kGlu as a constant)
// What a bf16 product over sorted pairs runs on.
struct ExpertForm {
  int rows, weights;           // of a tile
  bool second, one_block;      // (second: of the plan's tiles of 256 rows where it has both; one_block: no expert has more than 32 rows)
};
static ExpertForm expert_form(int64_t pairs, int experts, int N, int K, const ExpertLinearArgs::Shared& shared, bool wide_stores) {
  const int plan_rows = tile_rows(pairs, experts);
  ExpertForm f;
  f.second = plan_rows == 128 && wide_stores && large_tiles_pay(pairs, experts, N);
  f.rows = f.second ? 256 : plan_rows;
  const bool narrow = f.rows == 64 && narrow_pays(pairs, experts, N, K, shared);
  f.one_block = narrow && pairs <= 32 && shared.rows <= 32;
  f.weights = f.rows == 256 ? 256 : narrow ? 64 : 128;
  return f;
}

template <typename F> static void with_glu(int glu, F f) {
  if (glu == kClampedGlu) f(std::integral_constant<int, kClampedGlu>{});
  else if (glu == kSiluGlu) f(std::integral_constant<int, kSiluGlu>{});
  else f(std::integral_constant<int, kNoGlu>{});
}

static int expert_linear(void* out, int64_t out_row_stride, const void* x, int64_t x_row_stride, const void* w,
                         const int32_t* ids, void* plan, int64_t pairs, int experts, int N, int K, int per_token,
                         int glu, float alpha, float limit, float shift, const ExpertLinearArgs::Shared& shared, int dtype, void* stream) {
  if (dtype_size(dtype) == 0) return MVLLM_ERR_BAD_DTYPE;
  if (pairs < 0 || experts <= 0 || N <= 0 || K <= 0 || per_token < 0 || x_row_stride < K || out_row_stride < (glu ? N / 2 : N)) return MVLLM_ERR_BAD_SHAPE;
  if (dtype == MVLLM_F16 || experts > kMaxExperts || pairs > (1 << 30) || K % 64 != 0 || N % (glu ? 64 : 16) != 0 || x_row_stride % 8 != 0 ||
      out_row_stride % 4 != 0)
    return MVLLM_ERR_UNSUPPORTED;
  const int sh_N = shared.N, sh_K = shared.K;
  if (shared.rows != 0) {
    if (shared.rows < 0 || sh_N <= 0 || sh_K <= 0 || shared.x_stride < sh_K || shared.out_stride < (glu ? sh_N / 2 : sh_N)) return MVLLM_ERR_BAD_SHAPE;
    if (dtype != MVLLM_BF16 || glu == kClampedGlu || sh_K % 64 != 0 || sh_N % (glu ? 64 : 16) != 0 || shared.x_stride % 8 != 0 || shared.out_stride % 8 != 0 ||
        pairs == 0 || !plan)
      return MVLLM_ERR_UNSUPPORTED;
    const int64_t bytes = ((int64_t)(shared.rows - 1) * shared.x_stride + sh_K) * 2;
    if (bytes >= (int64_t)1 << 32 || (int64_t)sh_N * sh_K * 2 >= (int64_t)1 << 31) return MVLLM_ERR_UNSUPPORTED;
    if (!shared.x || !shared.w || !shared.out) return MVLLM_ERR_NULL_POINTER;
    if (!aligned16(shared.x) || !aligned16(shared.w) || !aligned16(shared.out)) return MVLLM_ERR_MISALIGNED;
  }
  if (pairs == 0) return MVLLM_OK;
  if (!out || !x || !w || (!plan && !ids)) return MVLLM_ERR_NULL_POINTER;
  if (!aligned16(out) || !aligned16(x) || !aligned16(w)) return MVLLM_ERR_MISALIGNED;
  if (!plan && (dtype != MVLLM_BF16 || pairs > kFewPairs)) return MVLLM_ERR_UNSUPPORTED;
  ExpertLinearArgs a = {};
  a.out = out; a.x = x; a.w = w; a.ids = ids; a.x_stride = x_row_stride; a.out_stride = out_row_stride; a.pairs = (int)pairs;
  a.experts = experts; a.N = N; a.K = K; a.per_token = per_token; a.alpha = alpha; a.limit = limit; a.shift = shift;
  a.shared = shared;
  a.shared.units = 1;
  if (shared.rows != 0) a.shared.x_bytes = (uint32_t)(((int64_t)(shared.rows - 1) * shared.x_stride + sh_K) * 2);
  hipStream_t s = (hipStream_t)stream;
  const int outputs = glu ? N / 2 : N;
  if (!plan) {
    const unsigned n32 = (unsigned)((outputs + 31) / 32), n64 = (unsigned)((outputs + 63) / 64), n_experts = (unsigned)experts;
    with_glu(glu, [&](auto G) {
      constexpr int kGlu = decltype(G)::value, kTiles = kGlu ? 2 : 4;
      const dim3 grid(kGlu ? n32 : n64, n_experts);
      if (K >= 2048) moe_linear_few_kernel<8, kGlu, kTiles><<<grid, dim3(512), 0, s>>>(a);
      else moe_linear_few_kernel<4, kGlu, kTiles><<<grid, dim3(256), 0, s>>>(a);
    });
    return launch_status();
  }
  const PlanArgs p = plan_parts_of(plan, ids, pairs, experts);
  a.sorted_pair = p.sorted_pair; a.row_start = p.row_start;
  if (dtype == MVLLM_BF16) {
    const ExpertForm form = expert_form(pairs, experts, N, K, shared, out_row_stride % 8 == 0);
    const int rows = form.rows, tile = form.weights;
    a.tile_expert = p.tiles[form.second].expert; a.tile_row = p.tiles[form.second].row; a.num_tiles = p.tiles[form.second].num;
    a.max_tiles = (int)max_tiles(pairs, experts, rows);
    a.n_tiles = (N + tile - 1) / tile;
    if (rows == 256 && out_row_stride % 8 != 0) return MVLLM_ERR_UNSUPPORTED;
    const int64_t x_rows = per_token ? (pairs + per_token - 1) / per_token : pairs, x_bytes = ((x_rows - 1) * x_row_stride + K) * 2;
    if (x_bytes >= (int64_t)1 << 32 || (int64_t)N * K * 2 >= (int64_t)1 << 31) return MVLLM_ERR_UNSUPPORTED;
    a.x_bytes = (uint32_t)x_bytes;
    if (shared.rows != 0) {
      a.shared.row_tiles = (shared.rows + rows - 1) / rows;
      a.shared.n_tiles = (sh_N + tile - 1) / tile;
      const int64_t tiles = 8 * (((int64_t)a.shared.row_tiles * a.shared.n_tiles + 7) / 8);
      if (tiles > 0x3fffffff) return MVLLM_ERR_BAD_SHAPE;
      a.shared.blocks = (int)tiles;
    }
    const int64_t blocks = 8 * (((int64_t)a.max_tiles * a.n_tiles + 7) / 8 + 1 + a.n_tiles) + a.shared.blocks;
    if (blocks > 0x7fffffff) return MVLLM_ERR_BAD_SHAPE;
    const bool own = K >= 4096 && large_tiles(pairs, experts, N) >= 640;         // (moe_linear_large_kernel)
    a.groups = (int)(own || blocks / 8 < kLargeGroups ? blocks / 8 : kLargeGroups);
    if (shared.rows != 0 && a.groups == kLargeGroups) a.shared.units = sh_K > K ? (sh_K + K / 2) / K : 1;
    a.token_factor = 0xffffffffu / (uint32_t)(per_token ? per_token : 1);
    with_glu(glu, [&](auto G) {
      constexpr int kGlu = decltype(G)::value;
      if (rows == 256) moe_linear_large_kernel<kGlu><<<dim3(8u * (unsigned)a.groups), dim3(256), 0, s>>>(a);
      else if (rows == 128) moe_linear_many_kernel<kGlu, 4><<<dim3((unsigned)blocks), dim3(256), 0, s>>>(a);
      else if (form.one_block) moe_linear_narrow_kernel<kGlu, 1><<<dim3((unsigned)blocks), dim3(256), 0, s>>>(a);
      else if (tile == 64) moe_linear_narrow_kernel<kGlu, 2><<<dim3((unsigned)blocks), dim3(256), 0, s>>>(a);
      else moe_linear_many_kernel<kGlu, 2><<<dim3((unsigned)blocks), dim3(256), 0, s>>>(a);
    });
  } else {
    int64_t z = pairs / (16 * (int64_t)experts) + 1;
    const dim3 grid((unsigned)(outputs / 16), (unsigned)experts, (unsigned)(z > 64 ? 64 : z));
    with_glu(glu, [&](auto G) { moe_linear_any_kernel<float, decltype(G)::value><<<grid, dim3(256), 0, s>>>(a); });
  }
  return launch_status();
}

extern "C" int mvllm_moe_linear_tiles(int64_t pairs, int experts, int N, int K, int shared_rows, int shared_N, int shared_K, int* rows, int* weight_rows) {
  if (pairs <= 0 || experts <= 0 || N <= 0 || K <= 0 || shared_rows < 0 || (shared_rows > 0 && (shared_N <= 0 || shared_K <= 0))) return MVLLM_ERR_BAD_SHAPE;
  ExpertLinearArgs::Shared shared = {};
  shared.rows = shared_rows; shared.N = shared_N; shared.K = shared_K;
  const ExpertForm f = expert_form(pairs, experts, N, K, shared, true);
  if (rows) *rows = f.one_block ? 32 : f.rows;
  if (weight_rows) *weight_rows = f.weights;
  return MVLLM_OK;
}

extern "C" int mvllm_moe_linear(void* out, int64_t out_row_stride, const void* x, int64_t x_row_stride, const void* w,
                                const int32_t* ids, void* plan, int64_t pairs, int experts, int N, int K, int per_token,
                                int glu, int dtype, void* stream) {
  return expert_linear(out, out_row_stride, x, x_row_stride, w, ids, plan, pairs, experts, N, K, per_token, glu ? kSiluGlu : kNoGlu,
                       0.f, 0.f, 0.f, ExpertLinearArgs::Shared{}, dtype, stream);
}

extern "C" int mvllm_moe_linear_shared(void* out, int64_t out_row_stride, const void* x, int64_t x_row_stride, const void* w, const int32_t* ids,
                                       void* plan, int64_t pairs, int experts, int N, int K, int per_token, int glu, void* shared_out,
                                       int64_t shared_out_row_stride, const void* shared_x, int64_t shared_x_row_stride, const void* shared_w,
                                       int shared_rows, int shared_N, int shared_K, int dtype, void* stream) {
  ExpertLinearArgs::Shared shared = {};
  shared.out = reinterpret_cast<bf16_t*>(shared_out); shared.x = reinterpret_cast<const bf16_t*>(shared_x); shared.w = reinterpret_cast<const bf16_t*>(shared_w);
  shared.out_stride = shared_out_row_stride; shared.x_stride = shared_x_row_stride; shared.rows = shared_rows; shared.N = shared_N; shared.K = shared_K;
  return expert_linear(out, out_row_stride, x, x_row_stride, w, ids, plan, pairs, experts, N, K, per_token, glu ? kSiluGlu : kNoGlu,
                       0.f, 0.f, 0.f, shared, dtype, stream);
}

extern "C" int mvllm_moe_linear_clamped(void* out, int64_t out_row_stride, const void* x, int64_t x_row_stride, const void* w,
                                        const int32_t* ids, void* plan, int64_t pairs, int experts, int N, int K,
                                        int per_token, float alpha, float limit, float shift, int dtype, void* stream) {
  return expert_linear(out, out_row_stride, x, x_row_stride, w, ids, plan, pairs, experts, N, K, per_token, kClampedGlu, alpha, limit,
                       shift, ExpertLinearArgs::Shared{}, dtype, stream);
}
