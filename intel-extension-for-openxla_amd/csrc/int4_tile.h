// Int4 weight-only GEMM on tiles of 64 to 128 rows (int4_tile.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace xmk {

struct Int4TileArgs {
  const _Float16* act;
  const uint32_t* qw;
  const _Float16* scales;
  const _Float16* zeros;
  const _Float16* bias;  // or null
  _Float16* out;
  int M, K, N, group;
  int row_blocks, col_blocks;  // (filled in by the launch)
};

// Whether the kernel takes the call: arguments that the entry points accept, of alignments and sizes its addressing covers.
bool int4_tile_applicable(const Int4TileArgs& p);
// The time the launch should take, in microseconds.
double int4_tile_cost(int64_t m, int64_t k, int64_t n, int64_t group);
void int4_tile_launch(const Int4TileArgs& p, hipStream_t st);

}  // namespace xmk
