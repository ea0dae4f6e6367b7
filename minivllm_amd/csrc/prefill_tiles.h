// Device helpers shared by the LDS-tiled prefill kernels (prefill_varlen.hip, prefill_pingpong.hip): 16-bit packing,
// row sums on the dot unit, the lane-xor-32 maximum, and the global -> LDS copy with its buffer descriptor.
#pragma once
#include <type_traits>
#include <utility>
#include "common.h"

namespace mvllm {

typedef __attribute__((ext_vector_type(4))) short v4s;
typedef __attribute__((ext_vector_type(2))) float v2f;
typedef __attribute__((ext_vector_type(2))) __bf16 v2bf16;
typedef __attribute__((ext_vector_type(2))) _Float16 v2f16;


// v_max3_f32 without the canonicalising self-max the compiler puts in front of every fmaxf operand that
// comes out of an MFMA (scores are finite or -inf here, never NaN).  The compiler does not know what the asm
// reads, so it does not space it from an MFMA that writes an operand: the caller has to order it after an
// ordinary instruction that reads the newest MFMA result.
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// max(x[l], x[l ^ 32]) in every lane l, by v_permlane32_swap.
__device__ __forceinline__ float max_with_lane_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  // r[0] = (x[0..31], x[0..31]), r[1] = (x[32..63], x[32..63]): their maximum is max(x[l], x[l ^ 32]) in every lane
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// x[l] + x[l ^ 32] in every lane l.
__device__ __forceinline__ float sum_with_lane_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Compile-time loop: f(std::integral_constant<int, 0>{}) ... f(std::integral_constant<int, N - 1>{}).
template <typename F, int... Is>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, Is...>) {
  (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

template <typename T> __device__ __forceinline__ uint32_t pack2(float a, float b);
template <> __device__ __forceinline__ uint32_t pack2<bf16_t>(float a, float b) {
  v2f x = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(x, v2bf16));
}
template <> __device__ __forceinline__ uint32_t pack2<f16_t>(float a, float b) {
  v2f x = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(x, v2f16));
}

// (lo, hi) of a packed 16-bit pair, each multiplied by c and rounded back to the element type.
template <typename T> __device__ __forceinline__ uint32_t scale_pair(uint32_t w, float c) {
  return pack2<T>(lo_to_float<T>(w) * c, hi_to_float<T>(w) * c);
}
// acc + lo + hi of a packed 16-bit pair in one instruction (v_dot2_f32_bf16 / v_dot2_f32_f16 against (1, 1)).
template <typename T> __device__ __forceinline__ float add_pair(uint32_t w, float acc);
template <> __device__ __forceinline__ float add_pair<bf16_t>(uint32_t w, float acc) {
  const v2bf16 ones = {(__bf16)1.0f, (__bf16)1.0f};
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2bf16, w), ones, acc, false);
}
template <> __device__ __forceinline__ float add_pair<f16_t>(uint32_t w, float acc) {
  const v2f16 ones = {(_Float16)1.0f, (_Float16)1.0f};
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(v2f16, w), ones, acc, false);
}

// 16 bytes per lane from a buffer resource (wave-uniform descriptor + per-lane 32-bit byte offset) straight
// into LDS at lds_base + 16 * lane (buffer_load_dwordx4 ... lds).  Lanes whose offset is at or past the
// descriptor's size read nothing and get zeros written, so tiles that run past the end of the tensor need no
// clamping.  Written as inline asm on purpose: the compiler then neither tracks the transfer in vmcnt nor
// inserts a full vmcnt(0) wait before the next LDS read, so the copy of tile j+1 really overlaps the math on
// tile j; completion is awaited explicitly with dma_wait_all() before the barrier.  No "memory" clobber: the
// destination buffer is not touched by ordinary code until after that wait and barrier (which do clobber), and
// a clobber here would pin every LDS read of the tile in flight to its side of the copy.
typedef __attribute__((ext_vector_type(4))) int v4i;
template <int LDS_IMM>   // LDS destination = lds_base + LDS_IMM: one scalar register serves all copies of a wave
__device__ __forceinline__ void dma16_to_lds(v4i rsrc, uint32_t lane_off, uint32_t lds_base) {
  asm volatile("s_add_u32 m0, %0, %3\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds_base), "v"(lane_off), "s"(rsrc), "n"(LDS_IMM) : "scc", "m0");
}
// The same with one more offset for all lanes (it counts in the bounds check); NT: lines that are read once.
template <int LDS_IMM, bool NT = false>
__device__ __forceinline__ void dma16_to_lds_at(v4i rsrc, uint32_t lane_off, uint32_t wave_off, uint32_t lds_base) {
  if constexpr (NT)
    asm volatile("s_add_u32 m0, %0, %4\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds" ::"s"(lds_base), "v"(lane_off), "s"(rsrc), "s"(wave_off), "n"(LDS_IMM) : "scc", "m0");
  else
    asm volatile("s_add_u32 m0, %0, %4\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds_base), "v"(lane_off), "s"(rsrc), "s"(wave_off), "n"(LDS_IMM) : "scc", "m0");
}
// The same from a 64-bit address per lane (no bounds check).
__device__ __forceinline__ void dma16_to_lds_from(const void* p, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_base), "v"(p) : "m0");
}
// Raw buffer descriptor: 48-bit base, stride 0, size in bytes, 32-bit untyped data.
__device__ __forceinline__ v4i make_rsrc(const char* base, uint32_t bytes) {
  const uint64_t b = (uint64_t)base;
  v4i r;
  r[0] = (int)(uint32_t)b;
  r[1] = (int)((uint32_t)(b >> 32) & 0xffffu);
  r[2] = (int)bytes;
  r[3] = 0x00020000;
  return r;
}
__device__ __forceinline__ void dma_wait_all() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// All but the N newest copies (nothing else of the wave may be in flight: loads count too).
template <int N>
__device__ __forceinline__ void dma_wait_but() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// A barrier that leaves copies in flight (__syncthreads waits for every one): this wave's LDS reads are complete.
__device__ __forceinline__ void workgroup_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

// The cache store of a packed batch as workgroups of the attention's own launch, behind its items: nothing there reads the cache, so neither waits for the
// other.  As a launch of its own the copy of a short batch's rows is 2.5 us of launch and 1 of copying, and as much again of the host's
// time, in front of a kernel that leaves most CUs idle.  us with the store in front / beside, bf16, 8 kv heads of 128: 7 prompts of 60 to 151,
// 32 heads, 12.4 / 8.4; 3 of 165 to 1036 24.0 / 20.2, one of 1800 40.2 / 36.9; 16 heads, 13 of 60 to 500 20.5 / 15.3, two of 900 to 1500 31.4 / 26.7;
// heads of 64, 16 of 250 20.2 / 16.4; fp32 one of 400 26.1 / 22.6, 8 of 18 to 305 27.6 / 23.4.  The two-group kernel has every CU to
// itself until its first workgroups are done: two of 2500, 16 heads 69.4 / 62.7, 32 heads, 4 of 1200 to 1800 83.9 / 79.3, 16 of 64 to 2048 143.8 / 143.2.
// Workgroups of the attention kernel's kThreads threads, 32 or 64 KB each; more than kStoreGroups would queue for the places that its LDS leaves.
constexpr unsigned kStoreGroups = 256;
template <int kThreads> __device__ __forceinline__ void store_beside(const StoreBeside& a) {
  typedef uint32_t unit __attribute__((ext_vector_type(4)));
  const unit *key = reinterpret_cast<const unit*>(a.key), *value = reinterpret_cast<const unit*>(a.value);
  unit *to_k = reinterpret_cast<unit*>(a.k_cache), *to_v = reinterpret_cast<unit*>(a.v_cache);
  const unsigned block = (blockIdx.x - a.first) * gridDim.y + blockIdx.y, blocks = (gridDim.x - a.first) * gridDim.y;
  for (unsigned at = block * 4 * kThreads + threadIdx.x; at < a.units; at += blocks * 4 * kThreads) {      // (units are below 2^30)
    unit k[4], v[4];
    int64_t to[4];
    static_for<4>([&](auto J) {
      constexpr int j = decltype(J)::value;
      const unsigned i = at + kThreads * j, in = i < a.units ? i : a.units - 1, row = in / a.row_units;
      const int64_t slot = a.slots[row];
      to[j] = i < a.units && slot >= 0 && slot < a.num_slots ? slot * a.row_units + (in - row * a.row_units) : -1;
      k[j] = key[in];
      v[j] = value[in];
    });
    static_for<4>([&](auto J) {
      constexpr int j = decltype(J)::value;
      if (to[j] >= 0) {
        to_k[to[j]] = k[j];
        to_v[to[j]] = v[j];
      }
    });
  }
}
// behind a grid of items, (x, ranges)
inline void add_store_groups(StoreBeside& a, dim3& grid) {
  a.first = grid.x;
  if (a.k_cache == nullptr) return;
  const unsigned all = (a.units + 1023) / 1024, n = all < kStoreGroups ? all : kStoreGroups;
  grid.x += (n + grid.y - 1) / grid.y;
}
// false: more rows than 32-bit positions reach, or rows that are not whole units
inline bool store_to(StoreBeside& a, const void* k, const void* v, void* k_cache, void* v_cache, const int64_t* slots, int64_t num_slots,
                     int64_t tokens, int64_t row_bytes) {
  if (row_bytes % 16 != 0 || row_bytes / 16 >= ((int64_t)1 << 30) || tokens * (row_bytes / 16) >= ((int64_t)1 << 30)) return false;
  a.row_units = (unsigned)(row_bytes / 16); a.units = (unsigned)(tokens * (row_bytes / 16));
  a.key = k; a.value = v; a.k_cache = k_cache; a.v_cache = v_cache; a.slots = slots; a.num_slots = num_slots;
  return true;
}

}  // namespace mvllm
