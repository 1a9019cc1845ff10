// Which output tile a work-group of the GEMM kernels takes.
//
// Consecutive blocks land on different XCDs (eight of them, each with its own L2), so each XCD gets a contiguous run of
// tiles, and a run walks the tiles in groups of some tile rows, so that it uses few rows of A and columns of B: about as
// many of the one as of the other, up to eight rows.  Microseconds against runs only where the tiles divide by eight, always
// in eight rows: 85 x 4001 x 2231 19.2 -> 12.5, 141 x 1280 x 7168 17.1 -> 13.6, 811 x 3488 x 4144 50 -> 40, 2244 x 9235 x 13131
// 1077 -> 1017; 80 drawn sizes of 20 rows and more 4 % on average, 110 with k of 129 to 1300 3 %.
// The host works the order out, the divisors' reciprocals included, because a work-group sends its first loads when it knows
// its tile: with that, and all arguments in front of those loads asked for at once (request_first_args), 1400 drawn products
// take 3 % less (the smallest 5 %) than with divisions and rounds of argument loads in the kernel, and those of them that were
// slower than before the runs by more than 3 % are 17 instead of 100: 948 x 704 x 64 4.47 (before the runs), 4.87, 4.5.
#pragma once
#include <cstdint>

namespace gemm_impl {

struct TileOrder {
  // Block b takes number (b % 8) * xcd_step + min(b % 8, rest) + b / 8 * round_step of the tiles,
  uint32_t xcd_step, rest, round_step;
  // which are numbered by groups of `group` tiles (1 << shift tile rows; last_rows of them in group last_group), in a group
  // column by column.  inv_*: 2^32 over the divisor, rounded down (2^32 - 1 for 1).
  uint32_t group, inv_group, last_group, last_rows, inv_last;
  int shift;
};
struct TileAt {
  int m, n;
};

// n / d: inv is short of 2^32 / d by less than one, and the estimate of the quotient by at most one.
__host__ __device__ __forceinline__ uint32_t tile_quotient(uint32_t n, uint32_t d, uint32_t inv) {
  const uint32_t q = (uint32_t)(((uint64_t)n * inv) >> 32);
  return q + (n - q * d >= d ? 1 : 0);
}
__host__ __device__ __forceinline__ TileAt tile_at(uint32_t block, const TileOrder& o) {
  const uint32_t x = block & 7;
  const uint32_t number = x * o.xcd_step + (x < o.rest ? x : o.rest) + (block >> 3) * o.round_step;
  const uint32_t g = tile_quotient(number, o.group, o.inv_group), at = number - g * o.group;
  const bool last = g == o.last_group;
  const uint32_t rows = last ? o.last_rows : 1u << o.shift;
  const uint32_t col = last ? tile_quotient(at, o.last_rows, o.inv_last) : at >> o.shift;
  return {(int)((g << o.shift) + at - col * rows), (int)col};
}

inline uint32_t tile_inverse(uint32_t d) { return d == 1 ? 0xffffffffu : (uint32_t)((uint64_t{1} << 32) / d); }
// Contiguous runs per XCD, or consecutive tiles on consecutive XCDs.
inline TileOrder tile_numbers(uint32_t tiles, bool runs) {
  TileOrder o{};
  o.xcd_step = runs ? tiles / 8 : 1;
  o.rest = runs ? tiles % 8 : 0;
  o.round_step = runs ? 1 : 8;
  return o;
}
// Groups of 1 << shift tile rows, and one of what is left.
inline void tile_groups(TileOrder& o, uint32_t tiles_m, uint32_t tiles_n, int shift) {
  o.shift = shift;
  o.group = tiles_n << shift;
  o.last_group = tiles_m >> shift;
  o.last_rows = tiles_m - (o.last_group << shift);
  if (o.last_rows == 0) o.last_rows = 1;  // (there is no such group)
  o.inv_group = tile_inverse(o.group);
  o.inv_last = tile_inverse(o.last_rows);
}

inline TileOrder tile_order(uint32_t tiles_m, uint32_t tiles_n, int K) {
  const uint32_t tiles = tiles_m * tiles_n, run = (tiles + 7) / 8;
  // With k of 128 or less it is the output that takes the time, and neighbours on different XCDs write it faster (4305 x
  // 12736 x 64 46.0 against 44.5).
  TileOrder o = tile_numbers(tiles, tiles % 8 == 0 || K > 128);
  tile_groups(o, tiles_m, tiles_n, run >= 24 ? 3 : run >= 6 ? 2 : run >= 2 ? 1 : 0);
  return o;
}
// Tiles of a kernel that splits K over a work-group's waves: along the shorter side, so that a run covers few rows and
// columns of tiles.  But where a few tile columns and a long K come to a second round of up to 128 work-groups, column by
// column over all XCDs: the second round is then of rows that the first has brought into a cache.  2274 x 112 x 5128 28.2 ->
// 21.6 us, 4598 x 64 x 2752 16.0 -> 13.5, 4938 x 64 x 5568 29.3 -> 25.3; of 60 sizes with k of 2100 to 8900 the worst 16.7 -> 17.4
// (the tile rows no multiple of eight, so that a row's tiles are on two XCDs).  With a shorter K it is the other way round:
// 3032 x 80 x 1088 7.0 against 8.5; with two tile columns the two are level at about 1300, with four at 2100.
inline TileOrder tile_order_slices(uint32_t tiles_m, uint32_t tiles_n, int K) {
  const uint32_t tiles = tiles_m * tiles_n;
  const bool again = tiles_m > tiles_n && tiles_n <= 4 && tiles > 256 && tiles <= 384 && K > 512 * ((int)tiles_n + 1);
  TileOrder o = tile_numbers(tiles, !again && (tiles % 8 == 0 || K > 128));
  tile_groups(o, tiles_m, tiles_n, 0);
  if (again || tiles_m <= tiles_n) {  // column by column: one group of all rows
    o.group = tiles;
    o.last_group = 0;
    o.last_rows = tiles_m;
    o.inv_group = tile_inverse(tiles);
    o.inv_last = tile_inverse(tiles_m);
  }
  return o;
}

}  // namespace gemm_impl
