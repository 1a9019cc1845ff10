// Instantiates the fp32 GEMM; see gemm_split.h.
#include "gemm_split.h"

namespace gemm_impl {
template <>
void launch_ragged<float, true>(bool a_mc, bool b_mc, GemmParams& p, int batch, int tile, hipStream_t st) {
  if (!a_mc && !b_mc) launch_f32_tile<false, false>(p, batch, tile, st);
  else if (!a_mc && b_mc) launch_f32_tile<false, true>(p, batch, tile, st);
  else if (a_mc && !b_mc) launch_f32_tile<true, false>(p, batch, tile, st);
  else launch_f32_tile<true, true>(p, batch, tile, st);
}
}  // namespace gemm_impl
