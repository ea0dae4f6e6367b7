// Prefill over a paged cache (16-bit, or INT8 codes with fp32 scales) with the keys of every sequence cut into ranges: a batch of few new tokens behind
// long cached prefixes (a follow-up turn of a chat, the last chunk of a chunked prefill) has too few query tiles to
// occupy the chip, and every one of them walks the whole prefix.  Here a sequence's prefix is cut into `splits - 1`
// ranges of whole key tiles and whole cache blocks plus one last range that holds the rest of the prefix and the new
// tokens; the one-group kernel of prefill_mfma.h walks each range as a sequence of its own (same queries, a block table
// that starts at the range's first block, every key of a prefix range visible, the last range causal) and writes a
// partial result and the logarithm of its softmax denominator per (query row, head); a second kernel merges them.
// Three launches: the plan (tables and offsets of the ranges, from lengths that only the device holds), the attention
// kernel, the merge.  No counterpart in the reference (its Triton prefill never reads the paged cache,
// attention.py:111-209).
#include <algorithm>

#include "common.h"
#include "prefill_mfma.h"

namespace mvllm {

namespace {

constexpr int kMaxRanges = 64;         // ranges of all sequences together: one wave plans them, and the attention kernel
                                       // deals the work of at most 64 sequences heaviest first

struct SplitArgs {
  const int32_t* cu_seqlens_q;
  const int32_t* cu_seqlens_k;
  const int32_t* block_tables;
  int32_t* ws_cu_q;        // [ranges + 1]
  int32_t* ws_cu_k;        // [ranges + 1]
  int32_t* ws_q_pos;       // [ranges]
  int32_t* ws_table;       // [ranges, table_width]
  int num_seqs;
  int splits;
  int unit;                // keys: a common multiple of the key tile (64) and the block size
  int block_size;
  int max_num_blocks;
  int table_width;
  int total_q;
};

struct Range { int key0, keys, q_pos; };
// Range i of sequence s (range numbering: i * num_seqs + s).
__device__ __forceinline__ Range range_of(const SplitArgs& a, int s, int i) {
  const int n = a.cu_seqlens_q[s + 1] - a.cu_seqlens_q[s];
  const int kv = a.cu_seqlens_k[s + 1] - a.cu_seqlens_k[s];
  const int cached = max(kv - n, 0);
  const int units = cached / a.unit;                           // whole units of the prefix
  const int per = (units + a.splits - 2) / (a.splits - 1);     // units per prefix range
  Range r;
  if (i < a.splits - 1) {
    const int u0 = min(i * per, units), u1 = min((i + 1) * per, units);
    r.key0 = u0 * a.unit;
    r.keys = n > 0 ? (u1 - u0) * a.unit : 0;
    r.q_pos = r.keys;                                          // every query row sees the whole range
  } else {
    r.key0 = units * a.unit;
    r.keys = n > 0 ? kv - r.key0 : 0;
    r.q_pos = cached - r.key0;
  }
  return r;
}

// Workgroup v: the block table of range v; workgroup 0 also the offsets of all ranges.
__global__ __launch_bounds__(64) void split_plan_kernel(const SplitArgs a) {
  const int ranges = a.num_seqs * a.splits;
  const int lane = threadIdx.x;
  if (blockIdx.x == 0) {
    int keys = 0;
    if (lane < ranges) {
      const int i = lane / a.num_seqs, s = lane - i * a.num_seqs;
      const Range r = range_of(a, s, i);
      keys = r.keys;
      a.ws_q_pos[lane] = r.q_pos;
      a.ws_cu_q[lane] = i * a.total_q + a.cu_seqlens_q[s];
    }
    int sum = keys;                                            // inclusive scan over the wave
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(sum, d, 64);
      if (lane >= d) sum += up;
    }
    if (lane < ranges) a.ws_cu_k[lane + 1] = sum;
    if (lane == 0) {
      a.ws_cu_k[0] = 0;
      a.ws_cu_q[ranges] = a.splits * a.total_q;
    }
  }
  const int v = blockIdx.x;
  const int i = v / a.num_seqs, s = v - i * a.num_seqs;
  const Range r = range_of(a, s, i);
  const int b0 = r.key0 / a.block_size;
  const int nb = (r.keys + a.block_size - 1) / a.block_size;
  const int32_t* src = a.block_tables + (int64_t)s * a.max_num_blocks;
  int32_t* dst = a.ws_table + (int64_t)v * a.table_width;
  for (int b = lane; b < a.table_width; b += 64) dst[b] = b < nb && b0 + b < a.max_num_blocks ? src[b0 + b] : -1;
}

struct MergeArgs {
  void* out;               // [total_q, Hq, D]
  const void* part;        // [splits * total_q, Hq, D]
  const float* lse;        // [splits * total_q, Hq]
  const int32_t* cu_seqlens_q;
  const int32_t* ws_cu_k;
  const float* sink;       // [Hq] or null: one more exp(sink) in every row's denominator
  int num_seqs;
  int splits;
  int total_q;
  int num_heads;
  int head_dim;
};

// One workgroup per (query row, slice of floor(256 / (D / 8)) heads); a thread merges 8 output elements of one head.  out =
// sum_i 2^(lse_i - M) o_i / sum_i 2^(lse_i - M) over the ranges that hold keys, M their largest lse: o_i is range i's
// normalised result and 2^lse_i its softmax denominator, so the weights restore the numerators.  The denominators of
// the slice are fetched into LDS first, all at once (an empty range's as -inf, which weighs it out), so that the loop
// over the ranges has nothing to wait for but its own independent loads.
template <typename T>
__global__ __launch_bounds__(256) void split_merge_kernel(const MergeArgs a) {
  __shared__ float lse_s[kMaxRanges][64];
  const int t = blockIdx.x;
  const int chunks = a.head_dim / 8;               // 4 .. 32
  const int heads_here = 256 / chunks;             // 64 .. 8
  const int head0 = blockIdx.y * heads_here;
  int s = 0;
  while (s + 1 < a.num_seqs && a.cu_seqlens_q[s + 1] <= t) ++s;
  for (int idx = threadIdx.x; idx < a.splits * heads_here; idx += 256) {
    const int i = idx / heads_here, hh = idx - i * heads_here;
    const int v = i * a.num_seqs + s;
    float x = -INFINITY;
    if (head0 + hh < a.num_heads && a.ws_cu_k[v + 1] - a.ws_cu_k[v] > 0)
      x = a.lse[((int64_t)i * a.total_q + t) * a.num_heads + head0 + hh];
    lse_s[i][hh] = x;
  }
  __syncthreads();
  const int hh = threadIdx.x / chunks, c = threadIdx.x - hh * chunks;
  const int h = head0 + hh;
  if (hh >= heads_here || h >= a.num_heads) return;
  float top = -INFINITY;
  for (int i = 0; i < a.splits; ++i) top = fmaxf(top, lse_s[i][hh]);
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  float den = 0.f;
  const T* part = reinterpret_cast<const T*>(a.part) + ((int64_t)t * a.num_heads + h) * a.head_dim + 8 * c;
  const int64_t stride = (int64_t)a.total_q * a.num_heads * a.head_dim;     // one range's partial results
#pragma unroll 4
  for (int i = 0; i < a.splits; ++i) {
    const float x = lse_s[i][hh];
    const float w = x == -INFINITY ? 0.f : exp2f(x - top);
    // an empty range's rows were never written: read them (the memory is the workspace's) but weigh them by a select,
    // not a product, so that whatever bits they hold stay out
    const uint4 p = *reinterpret_cast<const uint4*>(part + i * stride);
    den += w;
    const uint32_t words[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      acc[2 * e] = w != 0.f ? fmaf(w, lo_to_float<T>(words[e]), acc[2 * e]) : acc[2 * e];
      acc[2 * e + 1] = w != 0.f ? fmaf(w, hi_to_float<T>(words[e]), acc[2 * e + 1]) : acc[2 * e + 1];
    }
  }
  if (a.sink != nullptr) den = add_sink(den, top, a.sink[h]);
  const float inv = den > 0.f ? 1.f / den : 0.f;
  uint4 o;
  o.x = pack2<T>(acc[0] * inv, acc[1] * inv);
  o.y = pack2<T>(acc[2] * inv, acc[3] * inv);
  o.z = pack2<T>(acc[4] * inv, acc[5] * inv);
  o.w = pack2<T>(acc[6] * inv, acc[7] * inv);
  *reinterpret_cast<uint4*>(reinterpret_cast<T*>(a.out) + ((int64_t)t * a.num_heads + h) * a.head_dim + 8 * c) = o;
}

// The merge behind prefill_ranges.hip, with fp32 partial results: a wave merges one query row's heads, 256 / D of them at a time; rows
// whose tile has one range are complete already.
struct RangeMergeArgs {
  void* out;               // [total_q, Hq, D]
  const float* part;       // [ranges, total_q, Hq, D]
  const float* lse;        // [ranges, total_q, Hq]
  const int32_t* cu_seqlens_q;
  const int32_t* cu_seqlens_k;   // null: packed
  const float* sink;
  int num_seqs, ranges, range_tiles, rows_per_tile, total_q, num_heads;
};
template <typename T, int D, int kKeys = 64>
__global__ __launch_bounds__(256) void range_merge_kernel(const RangeMergeArgs a) {
  constexpr int kHeads = 256 / D, kLanes = D / 4;  // heads of a wave, lanes of a head
  const int lane = threadIdx.x & 63, t = blockIdx.x;
  // the row's sequence: at most 64 of them, one per lane
  int lo = 0, end = 0x7fffffff;
  if (lane < a.num_seqs) {
    lo = a.cu_seqlens_q[lane];
    end = a.cu_seqlens_q[lane + 1];
  }
  const int s = __popcll(__ballot(end <= t));
  if (s >= a.num_seqs) return;                     // behind the last sequence
  const int start = __builtin_amdgcn_readlane(lo, s), len = __builtin_amdgcn_readlane(end, s) - start;
  const int kv = a.cu_seqlens_k ? a.cu_seqlens_k[s + 1] - a.cu_seqlens_k[s] : len, cached = max(kv - len, 0);
  const int last = min((t - start) / a.rows_per_tile * a.rows_per_tile + a.rows_per_tile, len) - 1;
  const int tiles = min((cached + last) / kKeys, (kv - 1) / kKeys) + 1;
  if (tiles <= a.range_tiles) return;
  const int n = min((tiles + a.range_tiles - 1) / a.range_tiles, a.ranges);
  const int h = (blockIdx.y * 4 + (threadIdx.x >> 6)) * kHeads + lane / kLanes, c = 4 * (lane % kLanes);
  if (h >= a.num_heads) return;
  const int64_t at = (int64_t)t * a.num_heads + h, pitch = (int64_t)a.total_q * a.num_heads;
  // the weights: a range per lane of the head's, then through LDS (a wave's own: no barrier)
  __shared__ float weights[4 * kHeads][kMaxRanges];
  float* w_of = weights[(threadIdx.x >> 6) * kHeads + lane / kLanes];
  float lse[kMaxRanges / kLanes], top = -INFINITY;
#pragma unroll
  for (int j = 0; j < kMaxRanges / kLanes; ++j) {
    const int i = lane % kLanes + kLanes * j;
    lse[j] = i < n ? a.lse[i * pitch + at] : -INFINITY;
    top = fmaxf(top, lse[j]);
  }
#pragma unroll
  for (int o = 1; o < kLanes; o <<= 1) top = fmaxf(top, __shfl_xor(top, o, 64));
#pragma unroll
  for (int j = 0; j < kMaxRanges / kLanes; ++j) w_of[lane % kLanes + kLanes * j] = exp2f(lse[j] - top);
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  float den = 0.f;
#pragma unroll 8
  for (int i = 0; i < n; ++i) {
    const float w = w_of[i];
    const float4 p = *reinterpret_cast<const float4*>(a.part + (i * pitch + at) * D + c);
    den += w;
    acc.x = fmaf(w, p.x, acc.x);
    acc.y = fmaf(w, p.y, acc.y);
    acc.z = fmaf(w, p.z, acc.z);
    acc.w = fmaf(w, p.w, acc.w);
  }
  if (a.sink != nullptr) den = add_sink(den, top, a.sink[h]);
  const float inv = 1.f / den;
  if constexpr (std::is_same_v<T, float>)
    *reinterpret_cast<float4*>(reinterpret_cast<float*>(a.out) + at * D + c) = make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
  else
    *reinterpret_cast<uint2*>(reinterpret_cast<T*>(a.out) + at * D + c) =
        make_uint2(pack2<T>(acc.x * inv, acc.y * inv), pack2<T>(acc.z * inv, acc.w * inv));
}

int gcd_int(int x, int y) {
  while (y != 0) {
    const int r = x % y;
    x = y;
    y = r;
  }
  return x;
}

struct SplitLayout {
  int unit;
  int table_width;
  size_t ints_bytes;       // offsets, positions and tables, rounded up to 256
  size_t part_bytes;       // partial results, rounded up to 256
  size_t total_bytes;
};
SplitLayout split_layout(int num_seqs, int64_t total_q, int max_kv_len, int num_heads, int head_dim, int block_size, int splits) {
  SplitLayout l;
  l.unit = block_size / gcd_int(block_size, 64) * 64;
  const int ranges = num_seqs * splits;
  const int64_t units = max_kv_len / l.unit;
  const int64_t per = (units + splits - 2) / (splits - 1);
  const int64_t prefix_keys = per * l.unit;                                  // longest prefix range
  const int64_t last_keys = std::min<int64_t>(max_kv_len, l.unit + total_q); // longest last range
  l.table_width = (int)((std::max(prefix_keys, last_keys) + block_size - 1) / block_size) + 1;
  const size_t ints = (size_t)(2 * (ranges + 1) + ranges) + (size_t)ranges * l.table_width;
  l.ints_bytes = (ints * sizeof(int32_t) + 255) / 256 * 256;
  l.part_bytes = ((size_t)splits * total_q * num_heads * head_dim * 2 + 255) / 256 * 256;
  const size_t lse_bytes = ((size_t)splits * total_q * num_heads * sizeof(float) + 255) / 256 * 256;
  l.total_bytes = l.ints_bytes + l.part_bytes + lse_bytes;
  return l;
}

// int8: an INT8 cache (head_dim 64 and 128 only; a 16-bit cache also the other head dims of the LDS-tiled kernel)
bool split_shape_ok(int num_seqs, int64_t total_q, int max_kv_len, int num_heads, int num_kv_heads, int head_dim,
                    int block_size, int dtype, int splits, bool int8) {
  if (num_seqs <= 0 || total_q <= 0 || max_kv_len <= 0 || num_heads <= 0 || num_kv_heads <= 0 || block_size <= 0) return false;
  if (num_heads % num_kv_heads != 0 || num_heads > 65535) return false;
  if (dtype != MVLLM_BF16 && dtype != MVLLM_F16) return false;
  const bool dim_ok = head_dim == 128 || head_dim == 64 || (!int8 && prefill_mfma_other_dim(head_dim));
  if (!dim_ok || block_size % 16 != 0 || block_size > (1 << 20)) return false;
  if ((int64_t)block_size * num_kv_heads * head_dim * (int8 ? 1 : 2) >= ((int64_t)1 << 31)) return false;
  if (splits < 2 || (int64_t)num_seqs * splits > kMaxRanges) return false;
  if ((int64_t)splits * total_q > ((int64_t)1 << 30)) return false;
  return true;
}

}  // namespace

}  // namespace mvllm

using namespace mvllm;

// How many ranges to cut every sequence's keys into for a batch of these sizes (total_q_tokens new tokens in num_seqs
// sequences, the longest of max_kv_len keys): 0 = do not split (enough query tiles to fill the chip, keys too few to be
// worth the two extra launches, or a shape the split form is not built for).  The numbers: the two-group kernel deals
// items of 64 rows x 4 heads to 256 compute units, and a launch of fewer than 192 of them leaves a quarter of the chip
// idle from the start (shapes it does not take: fewer than three quarters of the one-group kernel's 512 places, 256 at head_dim 256);
// the one-group kernel that walks the ranges runs two workgroups per compute unit, so the ranges
// aim at 512 workgroups in all (but at 4 prefix ranges at least), each prefix range at least 1024 keys long, at most 16
// of them (more only lengthen the merge).
extern "C" int mvllm_prefill_paged_split_plan(int num_seqs, int64_t total_q_tokens, int max_kv_len, int num_heads,
                                              int num_kv_heads, int head_dim, int block_size, int dtype, int int8_cache) {
  if (!split_shape_ok(num_seqs, total_q_tokens, max_kv_len, num_heads, num_kv_heads, head_dim, block_size, dtype, 2, int8_cache != 0))
    return 0;
  if (max_kv_len < 4096) return 0;
  const int group = num_heads / num_kv_heads;
  const int hpw = group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
  const int rows = 32 * (4 / hpw);                    // query rows of a one-group workgroup
  // one-group workgroups of one range (every sequence but one may add a partial row tile)
  const int64_t items = ((total_q_tokens + rows - 1) / rows + num_seqs - 1) * (num_heads / hpw);
  const int places = head_dim == 256 ? 256 : 512;     // workgroups of the one-group kernel the chip holds at a time
  // what the call would run on otherwise: the two-group kernel (for an INT8 cache behind the staging step), or the
  // one-group kernel with its 512 places
  if (prefill_pp_takes(num_seqs, num_heads, num_kv_heads, head_dim, dtype, 16)) {
    const int64_t wide_items = (total_q_tokens / 64 + num_seqs) * std::max(num_heads / 4, 1);
    // INT8: the ranges run on the one-step kernel, which converts every tile for every query tile (two thirds of the
    // two-step form's rate), so the chip has to be emptier for the cut to pay (2 x 512 tokens behind 16384: 362 us in
    // two steps, 406 us cut)
    if (wide_items >= (int8_cache != 0 ? 96 : 192)) return 0;
  } else if (items >= 3 * places / 4) {
    return 0;
  }
  int64_t prefix_ranges = std::max<int64_t>(places / items - 1, 4);   // 4: a batch this small gains from any cut (measured)
  prefix_ranges = std::min<int64_t>(prefix_ranges, max_kv_len / 1024);
  prefix_ranges = std::min<int64_t>(prefix_ranges, kMaxRanges / num_seqs - 1);
  prefix_ranges = std::min<int64_t>(prefix_ranges, 16);
  return prefix_ranges >= 2 ? (int)prefix_ranges + 1 : 0;
}

extern "C" size_t mvllm_prefill_paged_split_workspace_bytes(int num_seqs, int64_t total_q_tokens, int max_kv_len, int num_heads,
                                                            int num_kv_heads, int head_dim, int block_size, int dtype, int splits) {
  if (!split_shape_ok(num_seqs, total_q_tokens, max_kv_len, num_heads, num_kv_heads, head_dim, block_size, dtype, splits, false)) return 0;
  return split_layout(num_seqs, total_q_tokens, max_kv_len, num_heads, head_dim, block_size, splits).total_bytes;
}

static int run_split(void* out, const void* q, const void* k_cache, const void* v_cache, const float* k_scale,
                     const float* v_scale, bool int8, const int32_t* block_tables, int max_num_blocks,
                     const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int num_seqs, int64_t total_q_tokens,
                     int max_kv_len, int num_heads, int num_kv_heads, int head_dim, int block_size, int64_t num_blocks,
                     float scale, const float* sink, int dtype, int splits, void* workspace, size_t workspace_bytes, void* stream) {
  if (dtype_size(dtype) == 0) return MVLLM_ERR_BAD_DTYPE;
  if (num_seqs < 0 || total_q_tokens < 0 || max_kv_len < 0 || num_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 ||
      block_size <= 0 || num_blocks < 0 || max_num_blocks < 0 || num_heads % num_kv_heads != 0 || !(scale > 0.f))
    return MVLLM_ERR_BAD_SHAPE;
  if (num_seqs == 0 || total_q_tokens == 0) return MVLLM_OK;
  if (!out || !q || !k_cache || !v_cache || (int8 && (!k_scale || !v_scale)) || !block_tables || !cu_seqlens_q || !cu_seqlens_k)
    return MVLLM_ERR_NULL_POINTER;
  if (!split_shape_ok(num_seqs, total_q_tokens, max_kv_len, num_heads, num_kv_heads, head_dim, block_size, dtype, splits, int8))
    return MVLLM_ERR_UNSUPPORTED;
  if (!aligned16(q) || !aligned16(out) || !aligned16(k_cache) || !aligned16(v_cache)) return MVLLM_ERR_MISALIGNED;
  const SplitLayout l = split_layout(num_seqs, total_q_tokens, max_kv_len, num_heads, head_dim, block_size, splits);
  if (!workspace || workspace_bytes < l.total_bytes || (reinterpret_cast<uintptr_t>(workspace) & 255u) != 0)
    return MVLLM_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  const int ranges = num_seqs * splits;
  int32_t* ints = reinterpret_cast<int32_t*>(workspace);
  SplitArgs sp;
  sp.cu_seqlens_q = cu_seqlens_q; sp.cu_seqlens_k = cu_seqlens_k; sp.block_tables = block_tables;
  sp.ws_cu_q = ints;
  sp.ws_cu_k = ints + (ranges + 1);
  sp.ws_q_pos = ints + 2 * (ranges + 1);
  sp.ws_table = ints + 2 * (ranges + 1) + ranges;
  sp.num_seqs = num_seqs; sp.splits = splits; sp.unit = l.unit; sp.block_size = block_size;
  sp.max_num_blocks = max_num_blocks; sp.table_width = l.table_width; sp.total_q = (int)total_q_tokens;
  split_plan_kernel<<<dim3((unsigned)ranges), dim3(64), 0, s>>>(sp);
  int status = launch_status();
  if (status != MVLLM_OK) return status;

  char* part = reinterpret_cast<char*>(workspace) + l.ints_bytes;
  float* lse = reinterpret_cast<float*>(part + l.part_bytes);
  PrefillArgs a;
  a.out = part; a.q = q; a.k = k_cache; a.v = v_cache; a.cu_seqlens = sp.ws_cu_q;
  a.total_tokens = (int64_t)splits * total_q_tokens; a.num_seqs = ranges; a.num_heads = num_heads;
  a.num_kv_heads = num_kv_heads; a.head_dim = head_dim; a.scale_log2 = scale * kLog2e;
  a.tiles_x = 0; a.heads_y = 0; a.band_bits = 0;
  a.cu_seqlens_k = sp.ws_cu_k; a.block_tables = sp.ws_table; a.max_num_blocks = l.table_width;
  a.block_size = block_size; a.num_blocks = num_blocks; a.k_scale = k_scale; a.v_scale = v_scale;
  a.q_pos = sp.ws_q_pos; a.lse = lse; a.q_period = total_q_tokens;
  status = int8                               ? launch_prefill_paged_int8(a, dtype, s)
           : prefill_mfma_other_dim(head_dim) ? launch_prefill_mfma_other(a, dtype, true, s)
                                              : launch_prefill_paged_16bit(a, dtype, s);
  if (status != MVLLM_OK) return status;

  MergeArgs m;
  m.out = out; m.part = part; m.lse = lse; m.cu_seqlens_q = cu_seqlens_q; m.ws_cu_k = sp.ws_cu_k;
  m.sink = sink;
  m.num_seqs = num_seqs; m.splits = splits; m.total_q = (int)total_q_tokens; m.num_heads = num_heads; m.head_dim = head_dim;
  const int heads_per_wg = 256 / (head_dim / 8);
  const dim3 grid((unsigned)total_q_tokens, (unsigned)((num_heads + heads_per_wg - 1) / heads_per_wg));
  if (dtype == MVLLM_BF16) split_merge_kernel<bf16_t><<<grid, dim3(256), 0, s>>>(m);
  else split_merge_kernel<f16_t><<<grid, dim3(256), 0, s>>>(m);
  return launch_status();
}

extern "C" int mvllm_prefill_paged_split(void* out, const void* q, const void* k_cache, const void* v_cache,
                                         const int32_t* block_tables, int max_num_blocks, const int32_t* cu_seqlens_q,
                                         const int32_t* cu_seqlens_k, int num_seqs, int64_t total_q_tokens, int max_kv_len,
                                         int num_heads, int num_kv_heads, int head_dim, int block_size, int64_t num_blocks,
                                         float scale, int dtype, int splits, void* workspace, size_t workspace_bytes,
                                         void* stream) {
  return run_split(out, q, k_cache, v_cache, nullptr, nullptr, false, block_tables, max_num_blocks, cu_seqlens_q, cu_seqlens_k,
                   num_seqs, total_q_tokens, max_kv_len, num_heads, num_kv_heads, head_dim, block_size, num_blocks, scale, nullptr, dtype,
                   splits, workspace, workspace_bytes, stream);
}

extern "C" int mvllm_prefill_paged_split_sink(void* out, const void* q, const void* k_cache, const void* v_cache,
                                              const int32_t* block_tables, int max_num_blocks, const int32_t* cu_seqlens_q,
                                              const int32_t* cu_seqlens_k, int num_seqs, int64_t total_q_tokens, int max_kv_len,
                                              int num_heads, int num_kv_heads, int head_dim, int block_size, int64_t num_blocks,
                                              float scale, const float* sink, int dtype, int splits, void* workspace,
                                              size_t workspace_bytes, void* stream) {
  return run_split(out, q, k_cache, v_cache, nullptr, nullptr, false, block_tables, max_num_blocks, cu_seqlens_q, cu_seqlens_k,
                   num_seqs, total_q_tokens, max_kv_len, num_heads, num_kv_heads, head_dim, block_size, num_blocks, scale, sink, dtype,
                   splits, workspace, workspace_bytes, stream);
}

extern "C" int mvllm_prefill_paged_int8_split(void* out, const void* q, const int8_t* k_cache, const int8_t* v_cache,
                                              const float* k_scale, const float* v_scale, const int32_t* block_tables,
                                              int max_num_blocks, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                                              int num_seqs, int64_t total_q_tokens, int max_kv_len, int num_heads,
                                              int num_kv_heads, int head_dim, int block_size, int64_t num_blocks, float scale,
                                              int dtype, int splits, void* workspace, size_t workspace_bytes, void* stream) {
  return run_split(out, q, k_cache, v_cache, k_scale, v_scale, true, block_tables, max_num_blocks, cu_seqlens_q, cu_seqlens_k,
                   num_seqs, total_q_tokens, max_kv_len, num_heads, num_kv_heads, head_dim, block_size, num_blocks, scale, nullptr, dtype,
                   splits, workspace, workspace_bytes, stream);
}

// ---- key ranges with their tables left where they are (prefill_ranges.hip) ----

// shapes the form takes: prefill_kernel_for's LDS-tiled kernel at head_dim 64 and 128, 64 sequences at most
static bool ranges_shape_ok(int num_seqs, int64_t total_q, int max_kv_len, int num_heads, int num_kv_heads, int head_dim, int block_size,
                            int dtype) {
  if (num_seqs <= 0 || num_seqs > 64 || total_q <= 0 || max_kv_len <= 0 || num_heads <= 0 || num_kv_heads <= 0 || block_size < 0) return false;
  if (num_heads % num_kv_heads != 0 || num_heads > 65535 || (dtype != MVLLM_BF16 && dtype != MVLLM_F16)) return false;
  if ((head_dim != 128 && head_dim != 64) || block_size % 16 != 0) return false;
  if ((int64_t)block_size * num_kv_heads * head_dim * 2 >= ((int64_t)1 << 31) || (int64_t)num_kv_heads * head_dim * 2 * 64 >= ((int64_t)1 << 31)) return false;
  return total_q <= ((int64_t)1 << 24);
}
static int rows_of_tile(int group) { return 32 * (group % 4 == 0 ? 1 : group % 2 == 0 ? 2 : 4); }
static int64_t ranges_of(int64_t max_kv_len, int64_t range_tiles) { return ((max_kv_len + 63) / 64 + range_tiles - 1) / range_tiles; }

// The busiest CU of a batch of equal sequences, in longest tiles: workgroup i of `wgs`, heaviest first within a sequence, lands on CU i
// mod 256 and costs 1 - fresh (place in its sequence), `fresh` being the share of the keys that the rows bring themselves.
static float busiest_cu(int64_t wgs, int num_seqs, float fresh) {
  const float of_seq = (float)wgs / (float)num_seqs;
  float most = 1.f;
  for (int64_t cu = 0; cu + 256 < wgs && cu < 256; ++cu) {
    float sum = 0.f;
    for (int64_t i = cu; i < wgs; i += 256) sum += 1.f - fresh * (fmodf((float)i, of_seq) / of_seq);
    most = fmaxf(most, sum);
  }
  return most;
}

// The range of a cached batch, which is even.  A workgroup alone on its CU waits a tile's trip to memory, 0.85 us, so that the longest sequence's chain
// decides until the CUs have several; `on_cu` is what a CU has in tiles, sequences of log-uniform lengths assumed, the more of them the further
// below the longest.  A merge takes 1.6 us and each range its partial results' way.  Fitted to 356 random batches, caches cold, and tried on 368 others: on
// average 1.4 % behind the best range of each (3.8 % before, where a range was at least 6 tiles and batches of more than 192 workgroups were whole).  1086
// batches, 1 to 16 sequences, took 0.977 of the time before, 192 of them less than 0.95, 14 more than 1.05 (five of 240 rows in all, 20 tiles, 16 heads 19.9 / 23.3;
// two of 554, 87 tiles 72.6 / 84; four of 480, 72 tiles, heads of 64 27.7 / 32).  us
// before / now, heads of 128: 12 of 755 rows in all, 95 % cached, 32 heads, up to 50 tiles 72.2 / 54; of 572, 37 tiles 55.4 / 38.9; three of 145, 16 tiles 23.2 /
// 17.9; furthest behind the best, nine of 12 tiles, 104 workgroups, 1.19 times as long.  From 193 workgroups on equal ones gain nothing (1500 rows behind 1500, 376
// workgroups: 72 whole, 86 in two), and few sequences may be equal.
struct CachedBatch {
  int64_t tiles;
  float on_cu, per_tile, start, wgs;       // wgs: workgroups of a range that have rows, were all sequences as long as their mean, or half of their last row tiles
};
static CachedBatch cached_batch(int num_seqs, int64_t total_q, int64_t max_kv_len, int num_heads, int num_kv_heads, int head_dim) {
  const int bm = rows_of_tile(num_heads / num_kv_heads);
  const int64_t slices = (int64_t)num_heads * bm / 128, tiles = ranges_of(max_kv_len, 1), wgs = (total_q / bm + num_seqs) * slices;
  const float fresh = fminf(1.f, (float)total_q / ((float)num_seqs * (float)max_kv_len)), of_seq = (float)total_q / (float)num_seqs / (float)bm;
  return {tiles, 1.29f * powf((float)num_seqs, -0.4f) * (1.f - 0.29f * fresh) * (float)(wgs * tiles) / 256.f, head_dim == 64 ? 0.58f : 0.85f,
          head_dim == 64 ? 0.8f : 2.f, fmaxf(ceilf(of_seq), of_seq + 0.5f) * (float)(num_seqs * slices)};
}
static float chain_us(const CachedBatch& b, int64_t x, bool pairs) {
  const float t = (float)x;
  return pairs ? b.start + b.per_tile * (0.85f * t + 0.3f * b.on_cu) : b.per_tile * (fmaxf(t, b.on_cu) + 0.7f * fminf(t, b.on_cu));
}
// Workgroups of two groups of four waves, each of which walks half of a range's tiles.  Alone on its CU a workgroup of one group takes 1.35 us per tile
// (870 rows behind 90 %, 14 tiles of 128 dims 18.5 us): products, softmax, LDS reads and trips to memory one after the other.  With two
// waves per SIMD they cover one another: 0.85 of the time per tile, for 0.8 (dims 64) or 2 us of a second group's start and of the sums' way through LDS.
// A workgroup takes most of a CU's LDS, so that it pays as long as each has a CU of its own.  Cached batches: the same model, fitted to 2700
// random ones of 7 tiles and more, 64 to 420 workgroups, caches warm: with the range that it chooses 1.047 times as fast as before on average, 2 % of them more
// than 3 % slower.  300 others of seven kinds of heads, 1 to 24 sequences: 1.036, between 0.953 and 1.269.  us before and now: one sequence of 451 rows,
// 141 tiles of 64 dims 42.8 / 35.4; two of 466, 73 tiles 42.0 / 36.7; three of 682, 26 tiles of 64 dims 23.8 / 20.3; one of 980, 31 tiles, 32 heads 46.9 / 42.1;
// but two of 2752, 67 tiles 113 / 117.  188 more, 30 to 97 % cached: 61 in two groups, 1.085 times as fast, one 0.929 (seven of 742 rows, 98 tiles 52.4 / 56.4).  Packed ones, whose row tiles differ, in 1000 batches: 13 to 16 tiles up to 256 workgroups 1.03 times as fast, 16 to 22 up to
// 320 1.07, 22 to 32 up to 400 1.04 to 1.14, 32 to 50 up to 480 1.15 to 1.24 (3071 rows, 64 dims 41.2 / 34.4); on the line's other side 10 to 13 tiles 0.99, 13 to
// 16 and 320 to 400 workgroups 0.92, 22 to 32 and 480 to 600 0.93.
static bool pairs_pay(int num_seqs, int64_t total_q, int64_t max_kv_len, int num_heads, int num_kv_heads, int head_dim, bool paged, int64_t range_tiles) {
  const CachedBatch b = cached_batch(num_seqs, total_q, max_kv_len, num_heads, num_kv_heads, head_dim);
  const int64_t x = std::min(range_tiles, b.tiles), n = (b.tiles + x - 1) / x;
  if (!paged) {
    const int bm = rows_of_tile(num_heads / num_kv_heads);
    const int64_t wgs = (total_q / bm + num_seqs) * ((int64_t)num_heads * bm / 128);
    return x >= 13 && (n == 1 ? wgs <= std::min<int64_t>(480, 256 + 11 * (x - 13)) : wgs * n <= 256);
  }
  return x >= 8 && b.wgs * (float)n <= 256.f && chain_us(b, x, true) + (n > 1 ? 1.f : 0.f) < chain_us(b, x, false);
}
// whole: what is not in pairs is one range.  apart: what is one range goes to another kernel, so that there is no pair of one either (taken for one, batches of
// 12 to 20 tiles of 64 dims lost their ranges: 552 rows behind as many 20.5 / 23.2 us, 324 behind 864, 16 heads 19.3 / 26.1).
static int64_t cached_range(const CachedBatch& b, float part_us, bool whole, bool apart) {
  const int64_t tiles = b.tiles;
  const float per_range = 0.6f + 0.81f * part_us;
  int64_t p = (tiles + 1) / 2 * 2;
  float best = 0.8f, best_pairs = 0.f;
  for (int64_t most = kMaxRanges; most >= 1; --most) {      // the shortest range that gives so many
    const int64_t even_tiles = ((tiles + most - 1) / most + 1) / 2 * 2, x = even_tiles < 4 ? 4 : even_tiles, n = (tiles + x - 1) / x;
    if (x >= tiles && most > 1) continue;
    const float us = n > 1 ? 1.6f + per_range * (float)n : 0.f, from = chain_us(b, tiles, false);
    const float gain = from - chain_us(b, x, false) - us;
    if (!whole && n > 1 && gain > best) {
      best = gain;
      p = x;
    }
    if (b.wgs * (float)n > 256.f || std::min(x, tiles) < 8 || (apart && n == 1)) continue;
    const float gain_pairs = from - chain_us(b, std::min(x, tiles), true) - us - (n > 1 ? 1.f : 0.f);
    if (gain_pairs > best_pairs && gain_pairs > best) {
      best = best_pairs = gain_pairs;
      p = x;
    }
  }
  return p;
}

// The range for a batch of these sizes, at least every sequence's tiles where none is cut; 0: the other kernels.
// Which kernel: the two-group kernel holds one workgroup per CU and runs faster once it has started (906 TFLOP/s against 680), but takes
// 6 us longer until then, and its longest item decides when there are few.  So this form takes what fits on the chip about at once, two
// workgroups per CU, and somewhat more where its many short row tiles meet the other's long ones: short prompts, and one prompt, whose tiles are all
// different.  All figures here are us there / here, bf16, captured layers with their store (beside packed prompts in either launch, in front of cached
// ones).  16 heads over 8 kv heads of 128: two prompts of 270 rows 16.0 / 9.8, one of 3600 (456 workgroups) 78 / 66, of 5800 (728) 142 / 135, 16 of 370 (864)
// 30.6 / 27.1, 13 of 430 (800) 31.6 / 26.7, but seven of 760 (720) 32.0 / 34.1, two of 2500 (640) 65 / 66; behind as many, 11 of 420 (664) 56 / 51, seven of 800
// (752) 80 / 82.  32 heads: nine of 120 (336) 11.3 / 10.2, 13 of 150 (584) 17.5 / 13.4, one of 1800 42 / 36, of 2500 (632) 62 / 58; of the limit's other side five of
// 530 (696) 25.8 / 24.4, six of 600 (944) 33.1 / 31.0, nine of 290 behind as many (720) 43.4 / 43.3, but four of 950 behind as many (976) 95 / 104, one of 2270 (568) 145 / 163.
// The two workgroups of a CU are the i-th and the (i + 256)-th.  Of a single sequence that is a heavy and a light one; of several equal
// ones it can be two of the heaviest, and the longer the tiles, the less the later start of the other kernel counts.  us, and busiest_cu: two prompts of
// 1496 (384 workgroups) 37.5 / 33.1 1.67, of 1656 (424) 40.5 / 38.8 1.79, of 1976 (504) 49.6 / 51.4 1.98, three of 976 (384) 28.3 / 28.2 2.0, of 1296 (504) 38.0 /
// 33.0 1.52; behind as many three of 794 rows (320) 51 / 47 1.80, four of 588 (320) 42.5 / 42.1 1.90; behind 95 %, nine of 128 (32 heads, 360)
// 64 / 74 2.0: the line lies a little low, by 4 % of one and nothing of the others.  Uneven ones meet by chance: 3300 rows of two (60 and 40 %) 46 / 36, of
// three 38 / 32.  Cached batches do not tell whether they are even and count as if.  With four heads per workgroup row tiles are half as long and equal
// sequences cost less: two prompts of 960 (496) 27.1 / 28.2, of 1040 30.5 / 31.1, three of 500 (392) 18.2 / 18.6, nine of 233 (592, busiest 3) 17.7 / 18.0, four of 680
// (712) 27.4 / 27.9, seven of 370 (696) 21.2 / 22.7; behind as many only two of them lose (of 815 51 / 52; four of 550 54 / 51).  (Above 112 tiles the other form
// cuts its keys too, and loses on either side of the line.)
// An odd head group has row tiles of 128 here as there, so that nothing is gained from shorter ones: packed batches lose (ten prompts of
// 332, 12 heads over 4: 15.9 / 16.6; five of 764, 14 over 2: 20.5 / 24.8; three of 400, 40 over 8, 480 places: 16.0 / 16.3), but where the other form's places of 256
// rows pass the chip's 512 and these workgroups do not (four of 280 19.5 / 14.0); cached ones gain what its empty places cost (seven of 55 rows behind as many, 40
// over 8: 19.7 / 14.9; ten of 163, 12 over 4, no empty places: 18.9 / 22.5) and where most keys are cached, so that tiles are alike (in the mean of 857 batches of
// random sizes, 1.2 times as fast; not ten of 163 behind 1467: 40 / 44); few workgroups with few keys gain nothing (two of 30 behind 270 13.4 / 13.3).
// At head_dim 64 the other form is this kernel over its banded order, 256 rows of a sequence at a time, the heaviest first: it pays for
// packed batches as soon as their tiles differ (3500 rows, 440 workgroups: 43.9 / 42.8; equal ones of a busiest CU above 1.5, three of 1925, 8
// heads, 26.0 / 34.7, of 1181, 12 heads over 4, 17.6 / 22.5).  Cached ones pay its empty places, which fill the
// chip's 512 the sooner; up to there its order gains where the CUs differ and most keys are not cached: two of 1852 rows
// behind as many, 16 heads (480 workgroups of 512 places, busiest 1.97) 69 / 76, three of 1266, 16 over 2 (480, 1.8) 48 / 52; four of 418
// of 758 keys, 32 heads (512 places) 21.7 / 22.0, of 350 (352 of 512) 20.3 / 22.6; with tiles of 64 or 128 rows a third of the places empty ends
// that (1.03 times as fast here in 40 random batches); beyond, of 518 of 958 (768) 29.0 / 27.3; eight of 93 of 168 (512 and 192) 12.6 / 11.1.
// With four heads per workgroup a band is eight tiles: packed batches of 400 to 600 workgroups gain where it has empty places (nine of 244 12.0 / 11.8,
// three of 600 15.9 / 14.5; two of 960, none empty, 16.0 / 19.8) or is one sequence (of 1800 24.2 / 23.8), cached ones up to 1400 (16 of
// 170 behind as many 27.7 / 22.2, three of 1600 behind 800 90 / 84; none empty: eight of 500 46 / 48).
// A few rows at head_dim 64 stay there, where placing the bands costs nothing (23 rows 4.8 / 4.8; five sequences of them, 32 heads, 5.2 / 4.9), and so do 200
// workgroups with more than 7000 keys, whose ranges the other form cuts (800 behind 7600, 32 heads of 128 141 / 144, of 64 94 / 109).
// Which range, packed (cached: cached_range): a tile takes a workgroup 0.9 us (0.8 at head_dim 64), workgroups of 0.6 of the longest sequence's tiles each fill 256 CUs;
// a range brings every row's fp32 partial result into memory and back, about 0.7 of the ranges are there on average.  Batches of more
// than 192 workgroups gain nothing that the partial results do not cost (1500 rows behind 1500, 32 heads, 376 workgroups: whole 72, two
// ranges 86).  The other kernels, split keys where they take them, / ranges: 343 rows behind 6500, 16 heads 50 / 43; 870 behind 7800 107 / 81; 132 of
// 32768, 32 heads 150 / 102.
extern "C" int mvllm_prefill_ranges_plan(int num_seqs, int64_t total_q_tokens, int max_kv_len, int num_heads, int num_kv_heads,
                                         int head_dim, int block_size, int dtype) {
  if (!ranges_shape_ok(num_seqs, total_q_tokens, max_kv_len, num_heads, num_kv_heads, head_dim, block_size, dtype)) return 0;
  const int group = num_heads / num_kv_heads, bm = rows_of_tile(group);
  const int64_t slices = (int64_t)num_heads * bm / 128, wgs = (total_q_tokens / bm + num_seqs) * slices, tiles = ranges_of(max_kv_len, 1);
  const bool four = group % 4 == 0, odd = group % 2 != 0, paged = block_size > 0;
  // were all sequences as long as their mean: workgroups that have rows, the other form's places
  const int64_t even = num_seqs * ((total_q_tokens + (int64_t)num_seqs * bm - 1) / ((int64_t)num_seqs * bm)) * slices;
  const int64_t places = num_seqs * ((total_q_tokens + (int64_t)num_seqs * 256 - 1) / ((int64_t)num_seqs * 256)) * (256 / bm) * slices;
  const bool packed64 = num_seqs == 1 ? even >= 384 && even <= 640 : num_seqs >= 3 && places > 512 && even >= 400 && even <= 600;
  const int64_t limit = head_dim == 64 ? (paged  ? (four && places > even ? 1400 : 768)
                                          : four ? (packed64 ? wgs : 0)
                                                 : tiles >= 16 ? 384 : 0)
                        : four  ? (paged && num_seqs == 1 ? 384 : 640)
                        : odd   ? (tiles >= 16 ? 512 : tiles >= 7 ? 580 : 640)
                        : paged ? (tiles >= 16 ? 512 : 780)
                                : (num_seqs == 1 ? 740 : tiles >= 16 ? 512 : tiles > 7 ? 580 : 980);
  if (wgs > limit) return 0;
  const float fresh = fminf(1.f, (float)total_q_tokens / ((float)num_seqs * (float)max_kv_len));
  const bool crowded = num_seqs > 1 && even > 272;
  if (head_dim == 64) {
    if (crowded && (paged ? fresh >= 0.3f && places <= 512 && (four || 10 * places <= 13 * even) : !four && fresh >= 0.75f) &&
        busiest_cu(even, num_seqs, fresh) > (paged ? 1.7f : 1.5f))
      return 0;
  } else {
    if (odd && !paged && (places <= 512 || even > 512 || total_q_tokens <= (int64_t)bm * num_seqs)) return 0;
    if (odd && paged && wgs > 192 && places <= 512 && 10 * places <= 11 * even && fresh >= 0.25f) return 0;
    if (crowded && tiles >= 16 && (paged ? tiles <= 112 && !(four && fresh >= 0.3f && num_seqs > 2) : fresh >= 0.87f) && busiest_cu(even, num_seqs, fresh) > (paged ? 1.85f : 1.75f)) return 0;
    if (four && crowded && !paged && fresh >= 0.87f && busiest_cu(even, num_seqs, fresh) > (num_seqs <= 3 ? 1.87f : 2.9f)) return 0;
  }
  int64_t p = (tiles + 1) / 2 * 2;
  const bool apart = wgs <= 192 && (head_dim == 64 ? wgs < (four ? 48 : 80) : odd && tiles < 8);
  if (paged)
    p = cached_range(cached_batch(num_seqs, total_q_tokens, max_kv_len, num_heads, num_kv_heads, head_dim),
                     8.f * (float)total_q_tokens * (float)(num_heads * head_dim) / 4.5e6f, wgs > 192 && num_seqs < 5, apart);
  if (wgs > 192) return (four || head_dim == 64) && tiles > 112 ? 0 : (int)p;
  const float per_tile = head_dim == 64 ? 0.8f : 0.9f, per_range = 0.3f + 0.7f * 8.f * (float)total_q_tokens * (float)(num_heads * head_dim) / 4.5e6f;
  float best = 3.f;
  for (int64_t most = kMaxRanges; !paged && most > 1; --most) {       // the shortest range that gives so many
    const int64_t even_tiles = ((tiles + most - 1) / most + 1) / 2 * 2, x = even_tiles < 6 ? 6 : even_tiles, n = (tiles + x - 1) / x;
    if (x >= tiles) continue;
    const float gain = per_tile * ((float)tiles - fmaxf((float)x, 0.6f * (float)(wgs * tiles) / 256.f)) - 4.f - per_range * (float)n;
    if (gain > best) {
      best = gain;
      p = x;
    }
  }
  return p >= tiles && apart ? 0 : (int)p;
}

extern "C" size_t mvllm_prefill_ranges_workspace_bytes(int64_t total_q_tokens, int max_kv_len, int num_heads, int head_dim, int range_tiles) {
  if (total_q_tokens <= 0 || max_kv_len <= 0 || num_heads <= 0 || head_dim <= 0 || range_tiles <= 0) return 0;
  const int64_t ranges = ranges_of(max_kv_len, range_tiles);
  return ranges < 2 ? 0 : (size_t)ranges * total_q_tokens * num_heads * (head_dim + 1) * sizeof(float);
}

extern "C" int mvllm_prefill_ranges_groups(int num_seqs, int64_t total_q_tokens, int max_kv_len, int num_heads, int num_kv_heads, int head_dim,
                                           int block_size, int dtype, int range_tiles) {
  if (range_tiles <= 0 || range_tiles % 2 != 0 ||
      !ranges_shape_ok(num_seqs, total_q_tokens, max_kv_len, num_heads, num_kv_heads, head_dim, block_size, dtype))
    return 0;
  return pairs_pay(num_seqs, total_q_tokens, max_kv_len, num_heads, num_kv_heads, head_dim, block_size > 0, range_tiles) ? 2 : 1;
}

static int run_ranges(void* out, const void* q, const void* k, const void* v, const int32_t* block_tables, int max_num_blocks,
                      const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int num_seqs, int64_t total_q_tokens, int max_kv_len,
                      int num_heads, int num_kv_heads, int head_dim, int block_size, int64_t num_blocks, float scale, const float* sink,
                      int dtype, int range_tiles, void* workspace, size_t workspace_bytes, const StoreBeside& store, void* stream) {
  if (dtype_size(dtype) == 0) return MVLLM_ERR_BAD_DTYPE;
  const bool paged = block_size > 0;
  if (num_seqs < 0 || total_q_tokens < 0 || max_kv_len < 0 || num_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 || block_size < 0 ||
      num_blocks < 0 || max_num_blocks < 0 || num_heads % num_kv_heads != 0 || !(scale > 0.f) || range_tiles <= 0)
    return MVLLM_ERR_BAD_SHAPE;
  if (num_seqs == 0 || total_q_tokens == 0) return MVLLM_OK;
  if (!out || !q || !k || !v || !cu_seqlens_q || (paged && (!block_tables || !cu_seqlens_k))) return MVLLM_ERR_NULL_POINTER;
  if (range_tiles % 2 != 0 || !ranges_shape_ok(num_seqs, total_q_tokens, max_kv_len, num_heads, num_kv_heads, head_dim, block_size, dtype))
    return MVLLM_ERR_UNSUPPORTED;
  if (ranges_of(max_kv_len, range_tiles) > kMaxRanges) return MVLLM_ERR_UNSUPPORTED;
  const int ranges = (int)ranges_of(max_kv_len, range_tiles);
  if (!aligned16(q) || !aligned16(out) || !aligned16(k) || !aligned16(v)) return MVLLM_ERR_MISALIGNED;
  if (ranges > 1 && (!workspace || !aligned16(workspace)) ||
      workspace_bytes < mvllm_prefill_ranges_workspace_bytes(total_q_tokens, max_kv_len, num_heads, head_dim, range_tiles))
    return MVLLM_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  PrefillArgs a = {};
  a.out = out; a.q = q; a.k = k; a.v = v; a.cu_seqlens = cu_seqlens_q; a.total_tokens = total_q_tokens; a.num_seqs = num_seqs;
  a.num_heads = num_heads; a.num_kv_heads = num_kv_heads; a.head_dim = head_dim; a.scale_log2 = scale * kLog2e;
  a.cu_seqlens_k = paged ? cu_seqlens_k : nullptr; a.block_tables = paged ? block_tables : nullptr; a.max_num_blocks = max_num_blocks;
  a.block_size = block_size; a.num_blocks = num_blocks; a.sink = sink;
  a.range_tiles = range_tiles;
  a.part = reinterpret_cast<float*>(workspace);
  a.lse = ranges > 1 ? a.part + (int64_t)ranges * total_q_tokens * num_heads * head_dim : nullptr;
  a.store = store;
  const int status = launch_prefill_ranges(a, dtype, paged, ranges, pairs_pay(num_seqs, total_q_tokens, max_kv_len, num_heads, num_kv_heads, head_dim, paged, range_tiles), s);
  if (status != MVLLM_OK || ranges == 1) return status;
  RangeMergeArgs m;
  m.out = out; m.part = a.part; m.lse = a.lse; m.cu_seqlens_q = cu_seqlens_q; m.cu_seqlens_k = a.cu_seqlens_k; m.sink = sink;
  m.num_seqs = num_seqs; m.ranges = ranges; m.range_tiles = range_tiles; m.rows_per_tile = rows_of_tile(num_heads / num_kv_heads);
  m.total_q = (int)total_q_tokens; m.num_heads = num_heads;
  const int per = 4 * (256 / head_dim);
  const dim3 grid((unsigned)total_q_tokens, (unsigned)((num_heads + per - 1) / per));
  if (dtype == MVLLM_BF16) {
    if (head_dim == 128) range_merge_kernel<bf16_t, 128><<<grid, dim3(256), 0, s>>>(m);
    else range_merge_kernel<bf16_t, 64><<<grid, dim3(256), 0, s>>>(m);
  } else {
    if (head_dim == 128) range_merge_kernel<f16_t, 128><<<grid, dim3(256), 0, s>>>(m);
    else range_merge_kernel<f16_t, 64><<<grid, dim3(256), 0, s>>>(m);
  }
  return launch_status();
}

extern "C" int mvllm_prefill_ranges(void* out, const void* q, const void* k, const void* v, const int32_t* block_tables,
                                    int max_num_blocks, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int num_seqs,
                                    int64_t total_q_tokens, int max_kv_len, int num_heads, int num_kv_heads, int head_dim, int block_size,
                                    int64_t num_blocks, float scale, const float* sink, int dtype, int range_tiles, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  return run_ranges(out, q, k, v, block_tables, max_num_blocks, cu_seqlens_q, cu_seqlens_k, num_seqs, total_q_tokens, max_kv_len, num_heads,
                    num_kv_heads, head_dim, block_size, num_blocks, scale, sink, dtype, range_tiles, workspace, workspace_bytes, StoreBeside{}, stream);
}

// ---- the same for fp32 (prefill_f32.hip), whose tiles are 32 keys ----

static bool f32_ranges_shape_ok(int num_seqs, int64_t total_q, int max_kv_len, int num_heads, int num_kv_heads, int head_dim, int block_size) {
  if (num_seqs <= 0 || num_seqs > 64 || total_q <= 0 || max_kv_len <= 0 || num_heads <= 0 || num_kv_heads <= 0 || block_size < 0) return false;
  if (num_heads % num_kv_heads != 0 || num_heads > 65535 || (head_dim != 128 && head_dim != 64) || block_size % 16 != 0) return false;
  if ((int64_t)num_kv_heads * head_dim * 4 * 64 >= ((int64_t)1 << 31) || (int64_t)block_size * num_kv_heads * head_dim * 4 >= ((int64_t)1 << 31)) return false;
  return total_q <= ((int64_t)1 << 24);
}
static int64_t f32_ranges_of(int64_t max_kv_len, int64_t range_tiles) { return ((max_kv_len + 31) / 32 + range_tiles - 1) / range_tiles; }

// The range for a batch of these sizes, all tiles where none is cut; 0: the kernel over whole rows.  A tile of 32 keys takes a workgroup 2.6 us
// at head_dim 64, 5.5 at 128, alone on its CU or in turns with another one, so what counts is how many tiles the busiest CU gets: `even` workgroups of equal
// sequences, the share of the longest one's tiles that they have on average, and 0.3 of a workgroup more where there are more than CUs or where
// the order has places without rows among them, two of which can meet.  The other order's places (256 rows of a sequence at a time) leave half of
// them empty from 128 rows per sequence down: 12 prompts of 60 rows behind 1100, 16 heads over 8 of 64 (96 workgroups of 384 places) 174 us there, 107 in this
// order uncut and 54 in 8 ranges; 16 of 100 behind 1900, 32 heads (512 workgroups) 425 and 300.  A merge is a launch (4 us) and
// the partial results' way through memory.  us whole and as planned, dims 64: 3 of 78 rows behind 1480, 16 heads 136 / 40; 20 behind 500
// 50 / 16; 40 behind 4000 331 / 30; one of 400, nothing cached, 36 / 23; 860 behind 860, 32 heads 148 / 115; two of 800 68 / 52, 32 heads
// 93, stay; 2000 behind 2000 (504 workgroups) 494 / 470; dims 128: 3 of 78 behind 1480 311 / 79, one of 2000 306 / 232.
extern "C" int mvllm_prefill_f32_ranges_plan(int num_seqs, int64_t total_q_tokens, int max_kv_len, int num_heads, int num_kv_heads,
                                             int head_dim, int block_size) {
  if (!f32_ranges_shape_ok(num_seqs, total_q_tokens, max_kv_len, num_heads, num_kv_heads, head_dim, block_size)) return 0;
  const int bm = rows_of_tile(num_heads / num_kv_heads);
  const int64_t slices = (int64_t)num_heads * bm / 128, tiles = f32_ranges_of(max_kv_len, 1), rows = (total_q_tokens + num_seqs - 1) / num_seqs;
  const int64_t even = num_seqs * ((rows + bm - 1) / bm) * slices, slots = (total_q_tokens / bm + num_seqs) * slices;
  const int64_t places = num_seqs * ((rows + 255) / 256) * (256 / bm) * slices;
  const float fresh = fminf(1.f, (float)total_q_tokens / ((float)num_seqs * (float)max_kv_len)), share = 1.f - 0.5f * fresh;
  const float tile = head_dim == 64 ? 2.6f : 5.5f, of_cus = (float)even / 256.f;
  const bool gaps = 10 * slots > 11 * even, padded = block_size > 0 && places > 256 && 2 * even <= places;
  auto busiest = [&](int64_t n) {                           // of n ranges, in ranges
    const bool meet = gaps && slots * n > 256;
    if (of_cus * (share * (float)n + 0.5f * fresh) <= 1.f && !meet) return 1.f;
    return fmaxf(1.f, 0.95f * share * of_cus * (float)n + (meet ? 0.6f : 0.3f));
  };
  const float whole = tile * (float)tiles * fmaxf(1.f, share * of_cus + (even > 256 ? 0.3f : 0.f)) * (padded ? 1.4f : 1.f);
  const float per_range = 0.3f + 0.7f * 8.f * (float)total_q_tokens * (float)(num_heads * head_dim) / 4.5e6f;
  float best = 0.93f * whole - 1.f;
  int64_t p = 0;
  if (padded && tile * (float)tiles * busiest(1) < best) {
    best = tile * (float)tiles * busiest(1);
    p = tiles;
  }
  if (padded && even > 256) return (int)p;
  for (int64_t most = tiles < kMaxRanges ? tiles : kMaxRanges; most > 1; --most) {
    const int64_t x = (tiles + most - 1) / most, n = (tiles + x - 1) / x;
    if (x < 2 || x >= tiles) continue;
    const float us = tile * (float)x * busiest(n) + 4.f + per_range * (float)n;
    if (us < best) {
      best = us;
      p = x;
    }
  }
  return (int)p;
}

extern "C" size_t mvllm_prefill_f32_ranges_workspace_bytes(int64_t total_q_tokens, int max_kv_len, int num_heads, int head_dim,
                                                           int range_tiles) {
  if (total_q_tokens <= 0 || max_kv_len <= 0 || num_heads <= 0 || head_dim <= 0 || range_tiles <= 0) return 0;
  const int64_t ranges = f32_ranges_of(max_kv_len, range_tiles);
  return ranges < 2 ? 0 : (size_t)ranges * total_q_tokens * num_heads * (head_dim + 1) * sizeof(float);
}

static int run_f32_ranges(float* out, const float* q, const float* k, const float* v, const int32_t* block_tables, int max_num_blocks,
                          const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int num_seqs, int64_t total_q_tokens, int max_kv_len,
                          int num_heads, int num_kv_heads, int head_dim, int block_size, int64_t num_blocks, float scale, const float* sink,
                          int range_tiles, void* workspace, size_t workspace_bytes, const StoreBeside& store, void* stream) {
  const bool paged = block_size > 0;
  if (num_seqs < 0 || total_q_tokens < 0 || max_kv_len < 0 || num_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 || block_size < 0 ||
      num_blocks < 0 || max_num_blocks < 0 || num_heads % num_kv_heads != 0 || !(scale > 0.f) || range_tiles <= 0)
    return MVLLM_ERR_BAD_SHAPE;
  if (num_seqs == 0 || total_q_tokens == 0) return MVLLM_OK;
  if (!out || !q || !k || !v || !cu_seqlens_q || (paged && (!block_tables || !cu_seqlens_k))) return MVLLM_ERR_NULL_POINTER;
  if (!f32_ranges_shape_ok(num_seqs, total_q_tokens, max_kv_len, num_heads, num_kv_heads, head_dim, block_size) ||
      f32_ranges_of(max_kv_len, range_tiles) > kMaxRanges)
    return MVLLM_ERR_UNSUPPORTED;
  const int ranges = (int)f32_ranges_of(max_kv_len, range_tiles);
  if (!aligned16(q) || !aligned16(out) || !aligned16(k) || !aligned16(v)) return MVLLM_ERR_MISALIGNED;
  if ((ranges > 1 && (!workspace || !aligned16(workspace))) ||
      workspace_bytes < mvllm_prefill_f32_ranges_workspace_bytes(total_q_tokens, max_kv_len, num_heads, head_dim, range_tiles))
    return MVLLM_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  PrefillArgs a = {};
  a.out = out; a.q = q; a.k = k; a.v = v; a.cu_seqlens = cu_seqlens_q; a.total_tokens = total_q_tokens; a.num_seqs = num_seqs;
  a.num_heads = num_heads; a.num_kv_heads = num_kv_heads; a.head_dim = head_dim; a.scale_log2 = scale * kLog2e;
  a.cu_seqlens_k = paged ? cu_seqlens_k : nullptr; a.block_tables = paged ? block_tables : nullptr; a.max_num_blocks = max_num_blocks;
  a.block_size = block_size; a.num_blocks = num_blocks; a.sink = sink;
  a.range_tiles = range_tiles;
  a.part = reinterpret_cast<float*>(workspace);
  a.lse = ranges > 1 ? a.part + (int64_t)ranges * total_q_tokens * num_heads * head_dim : nullptr;
  a.store = store;
  const int status = launch_prefill_f32_ranges(a, paged, ranges, s);
  if (status != MVLLM_OK || ranges == 1) return status;
  RangeMergeArgs m;
  m.out = out; m.part = a.part; m.lse = a.lse; m.cu_seqlens_q = cu_seqlens_q; m.cu_seqlens_k = a.cu_seqlens_k; m.sink = sink;
  m.num_seqs = num_seqs; m.ranges = ranges; m.range_tiles = range_tiles; m.rows_per_tile = rows_of_tile(num_heads / num_kv_heads);
  m.total_q = (int)total_q_tokens; m.num_heads = num_heads;
  const int per = 4 * (256 / head_dim);
  const dim3 grid((unsigned)total_q_tokens, (unsigned)((num_heads + per - 1) / per));
  if (head_dim == 128) range_merge_kernel<float, 128, 32><<<grid, dim3(256), 0, s>>>(m);
  else range_merge_kernel<float, 64, 32><<<grid, dim3(256), 0, s>>>(m);
  return launch_status();
}

extern "C" int mvllm_prefill_f32_ranges(float* out, const float* q, const float* k, const float* v, const int32_t* block_tables,
                                        int max_num_blocks, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int num_seqs,
                                        int64_t total_q_tokens, int max_kv_len, int num_heads, int num_kv_heads, int head_dim,
                                        int block_size, int64_t num_blocks, float scale, const float* sink, int range_tiles,
                                        void* workspace, size_t workspace_bytes, void* stream) {
  return run_f32_ranges(out, q, k, v, block_tables, max_num_blocks, cu_seqlens_q, cu_seqlens_k, num_seqs, total_q_tokens, max_kv_len, num_heads,
                        num_kv_heads, head_dim, block_size, num_blocks, scale, sink, range_tiles, workspace, workspace_bytes, StoreBeside{}, stream);
}

extern "C" int mvllm_prefill_store(void* out, const void* q, const void* k, const void* v, void* k_cache, void* v_cache,
                                   const int64_t* slot_mapping, int64_t num_slots, const int32_t* cu_seqlens, int num_seqs,
                                   int64_t total_tokens, int max_seqlen, int num_heads, int num_kv_heads, int head_dim, float scale,
                                   int dtype, int range_tiles, void* workspace, size_t workspace_bytes, void* stream) {
  if (dtype_size(dtype) == 0) return MVLLM_ERR_BAD_DTYPE;
  if (num_slots < 0 || total_tokens < 0 || num_kv_heads <= 0 || head_dim <= 0) return MVLLM_ERR_BAD_SHAPE;
  if (num_seqs == 0 || total_tokens > ((int64_t)1 << 30)) return MVLLM_ERR_UNSUPPORTED;          // (no sequences: there may be rows to store all the same)
  if (!k_cache || !v_cache || !slot_mapping) return MVLLM_ERR_NULL_POINTER;
  if (!aligned16(k_cache) || !aligned16(v_cache)) return MVLLM_ERR_MISALIGNED;
  StoreBeside to;
  if (!store_to(to, k, v, k_cache, v_cache, slot_mapping, num_slots, total_tokens, (int64_t)num_kv_heads * head_dim * dtype_size(dtype)))
    return MVLLM_ERR_UNSUPPORTED;
  if (range_tiles == 0)
    return run_prefill_varlen(out, q, k, v, cu_seqlens, num_seqs, total_tokens, num_heads, num_kv_heads, head_dim, scale, nullptr, dtype, to, stream);
  return dtype == MVLLM_F32
             ? run_f32_ranges((float*)out, (const float*)q, (const float*)k, (const float*)v, nullptr, 0, cu_seqlens, nullptr, num_seqs, total_tokens,
                              max_seqlen, num_heads, num_kv_heads, head_dim, 0, 0, scale, nullptr, range_tiles, workspace, workspace_bytes, to, stream)
             : run_ranges(out, q, k, v, nullptr, 0, cu_seqlens, nullptr, num_seqs, total_tokens, max_seqlen, num_heads, num_kv_heads, head_dim, 0, 0,
                          scale, nullptr, dtype, range_tiles, workspace, workspace_bytes, to, stream);
}
