// Instantiates the ragged MFMA GEMM for one (element type, output type) pair; see gemm_ragged.h.
#include "gemm_ragged.h"

namespace gemm_impl {
template <>
void launch_ragged<float, true>(bool a_mc, bool b_mc, GemmParams& p, int batch, int tile, hipStream_t st) {
  launch_ragged_impl<float, true>(a_mc, b_mc, p, batch, tile, st);
}
}  // namespace gemm_impl
