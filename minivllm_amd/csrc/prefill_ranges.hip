// The one-group prefill kernel (prefill_mfma.h) over ranges of key tiles, workgroups of a range side by side: for batches whose query
// tiles are too few to fill the chip, or so uneven that the longest one decides.  What a range of a row tile sees follows from the
// lengths in the workgroup itself, so nothing runs in front of the kernel; prefill_split.hip has the rule, the merge behind it and
// the entry points.
#include "prefill_mfma.h"

namespace mvllm {

template <typename T, bool PAGED>
static int launch(const PrefillArgs& a, int ranges, bool pairs, hipStream_t s) {
  return a.head_dim == 64 ? launch_prefill_mfma_as<T, PAGED, false, 64, 64, true>(a, s, ranges, pairs)
                          : launch_prefill_mfma_as<T, PAGED, false, 128, 128, true>(a, s, ranges, pairs);
}

int launch_prefill_ranges(const PrefillArgs& a, int dtype, bool paged, int ranges, bool pairs, hipStream_t s) {
  if (dtype == MVLLM_BF16) return paged ? launch<bf16_t, true>(a, ranges, pairs, s) : launch<bf16_t, false>(a, ranges, pairs, s);
  return paged ? launch<f16_t, true>(a, ranges, pairs, s) : launch<f16_t, false>(a, ranges, pairs, s);
}

}  // namespace mvllm
