// Instantiates the slices GEMM for one (element type, output type) pair; see gemm_slices.h.
#include "gemm_slices.h"

namespace gemm_impl {
template <>
void launch_slices<__bf16, false>(bool a_mc, bool b_mc, int v, GemmParams& p, int batch, hipStream_t st) {
  launch_slices_impl<__bf16, false>(a_mc, b_mc, v, p, batch, st);
}
}  // namespace gemm_impl
