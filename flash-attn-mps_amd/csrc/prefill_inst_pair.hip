// Wave-pair prefill variants: 256-dim heads, 16-bit K/V.
#include "prefill_pair.h"

namespace fa_prefill {

namespace {

template <typename T, bool CAUSAL>
PrefillKernel kernel(bool cap, bool win) {
  if (win) return cap ? prefill_pair_kernel<T, CAUSAL, true, true> : prefill_pair_kernel<T, CAUSAL, false, true>;
  return cap ? prefill_pair_kernel<T, CAUSAL, true, false> : prefill_pair_kernel<T, CAUSAL, false, false>;
}

}  // namespace

PrefillChoice pick_pair(bool bf16, bool causal, bool cap, bool win) {
  PrefillKernel k = bf16 ? (causal ? kernel<BF16T, true>(cap, win) : kernel<BF16T, false>(cap, win))
                         : (causal ? kernel<F16T, true>(cap, win) : kernel<F16T, false>(cap, win));
  return PrefillChoice{k, PAIR_ROWS, 64 * PAIR_WAVES, PAIR_LDS, 1};
}

}  // namespace fa_prefill
