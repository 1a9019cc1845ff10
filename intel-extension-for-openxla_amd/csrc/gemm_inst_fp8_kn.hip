// Instantiates the any-alignment kernels for fp8 with one storage order of B; see gemm_fp8.h.
#include "gemm_fp8.h"

namespace gemm_impl {
void launch_fp8_any_kn(int policy, Fp8Params& p, hipStream_t st) {
  if (policy >= kFp8Slices) launch_slices_rows<Fp8, false, false, true>(policy - kFp8Slices, p, 1, st);
  else launch_ragged_tile<Fp8, false, false, true>(p, 1, kFp8Policies[policy].bm, st);
}
}  // namespace gemm_impl
