// Fused multi-head attention forward, head sizes 65 to 80.
#include "fmha_fwd_kernel.h"

namespace fmha_fwd_impl {

void launch_h80(const FmhaParams& p, int32_t dtype, uint64_t units, uint32_t F, bool causal, int bias, hipStream_t st) {
  if (dtype == XMK_BF16) launch_cfg<__bf16, 128, 5, 3, 4, 2>(p, units, F, causal, bias, st);
  else launch_cfg<_Float16, 128, 5, 3, 4, 2>(p, units, F, causal, bias, st);
}

}  // namespace fmha_fwd_impl
