// The prefill_attn_kernel instances of soft-capped scores.
#include "prefill_attn.h"

namespace dlb {
void launch_prefill_capped(const PrefillParams& p, const PrefillForm& form, dim3 grid, hipStream_t s) {
  launch_prefill_kernel<true>(p, form, grid, s);
}
}  // namespace dlb
