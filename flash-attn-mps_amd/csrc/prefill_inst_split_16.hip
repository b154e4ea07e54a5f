// Key-split prefill variants with 16-bit K/V.
#include "prefill_kernel.h"

namespace fa_prefill {

PrefillChoice pick_split_16(bool bf16, int64_t dq, int64_t dv, bool causal, bool cap) {
  return bf16 ? pick_split<BF16T, BF16T, BF16T>(dq, dv, causal, cap)
              : pick_split<F16T, F16T, F16T>(dq, dv, causal, cap);
}

}  // namespace fa_prefill
