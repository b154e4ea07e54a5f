// Key-split prefill variants with E4M3 K/V.
#include "prefill_kernel.h"

namespace fa_prefill {

PrefillChoice pick_split_fp8(bool bf16, int64_t dq, int64_t dv, bool causal, bool cap) {
  return bf16 ? pick_split<BF16T, E4M3T, BF16T>(dq, dv, causal, cap)
              : pick_split<F16T, E4M3T, F16T>(dq, dv, causal, cap);
}

}  // namespace fa_prefill
