// Operand tiles for the kernels that take any alignment (gemm_ragged.h, gemm_slices.h): global memory -> registers
// -> LDS in 16-byte chunks, and the matrix-core fragments read back from LDS.
//
// A K step is 128 bytes of a reduction-contiguous row: 64 elements of 16 bits, 32 of fp32.
//   KC operand (reduction index contiguous): LDS [row][128 bytes], chunks XORed by pairs of rows.
//   MC operand (free index contiguous): LDS [k][rows], 16-bit elements read with the transpose loads, fp32 ones
//       as scalars.
// Every lane fetches whole chunks (the hardware takes global loads at any byte address), never element by
// element: a chunk that would reach past the end of its row is read from 16 bytes before that end and shifted
// into place, so nothing outside the matrix is touched and no lane branches.
#pragma once
#include "gemm_kernel.h"

namespace gemm_impl {

template <> struct Elem<float> {
  typedef floatx4 vec8;  // four consecutive k: operands of four matrix instructions
  static __device__ __forceinline__ float to_f32(float v) { return v; }
  static __device__ __forceinline__ uint16_t from_f32(float) { return 0; }  // fp32 outputs only
};

// v moved down by `bytes` (>= 0), zeros behind.
__device__ __forceinline__ u32x4 shift_bytes(u32x4 v, int bytes) {
  const int d = bytes >> 2;
  if (d & 1) v = u32x4{v[1], v[2], v[3], 0u};
  if (d & 2) v = u32x4{v[2], v[3], 0u, 0u};
  if (d & ~3) v = u32x4{0u, 0u, 0u, 0u};
  const uint32_t b = bytes & 3;
  return u32x4{__builtin_amdgcn_alignbyte(v[1], v[0], b), __builtin_amdgcn_alignbyte(v[2], v[1], b),
               __builtin_amdgcn_alignbyte(v[3], v[2], b), __builtin_amdgcn_alignbyte(0u, v[3], b)};
}

__device__ __forceinline__ u32x4 load16_any(const char* base, uint32_t off) {
  u32x4 v;
  __builtin_memcpy(&v, base + off, 16);  // one global_load_dwordx4 at any alignment
  return v;
}

// One operand tile of ROWS rows (or columns) x one K step, fetched by NT threads as NL chunks of 16 bytes each.
// Chunk i of thread t goes to LDS bytes [16 (i NT + t), +16).
template <typename T, bool MC, int ROWS, int NT>
struct AnyLoader {
  static constexpr int EB = sizeof(T), CE = 16 / EB, BK = 128 / EB;
  static constexpr int CPR = MC ? ROWS * EB / 16 : 8;  // chunks per LDS row
  static constexpr int RPL = NT / CPR;                 // LDS rows per load
  static constexpr int NL = ROWS * 8 / NT;
  static_assert(NL >= 1 && RPL % 4 == 0 && (MC || RPL % 8 == 0), "the swizzle repeats, or changes by element()'s term");
  uint32_t off[NL];  // byte offset of chunk i from the operand's K step origin
  int lrow, c0;      // LDS row and first element within that row of chunk 0
  int shift;         // MC: bytes by which the chunks were moved back to stay inside their rows

  static __device__ __forceinline__ int swizzle(int row_or_k) {
    if constexpr (MC && EB == 4) return 0;
    else return swz<MC, ROWS, 64>(row_or_k);
  }
  // First element of chunk i within its LDS row.  (KC: the XOR counts pairs of rows modulo 16 rows.)
  __device__ __forceinline__ int element(int i) const { return !MC && RPL % 16 != 0 && (i & 1) ? c0 ^ (4 * CE) : c0; }
  // row0: first row (KC) or column (MC) of the tile; rows: how many the matrix has (MC: at least CE).
  __device__ __forceinline__ void init(int64_t ld, int row0, int rows, int tid) {
    lrow = tid / CPR;
    c0 = ((tid % CPR) ^ swizzle(lrow)) * CE;
    shift = 0;
    if constexpr (MC) {
      const int col = row0 + c0, at = min(col, rows - CE);
      shift = (col - at) * EB;
#pragma unroll
      for (int i = 0; i < NL; ++i) off[i] = (uint32_t)(((int64_t)(lrow + i * RPL) * ld + at) * EB);
    } else {
#pragma unroll
      for (int i = 0; i < NL; ++i) {  // rows past the end repeat the last one: their products are not stored
        const int r = min(row0 + lrow + i * RPL, rows - 1) - row0;
        off[i] = (uint32_t)(((int64_t)r * ld + element(i)) * EB);
      }
    }
  }
  // base: the operand at this K step's first k (KC: of the tile's first row; MC: of column 0).
  __device__ __forceinline__ void load(const char* base, u32x4 (&g)[NL]) const {
#pragma unroll
    for (int i = 0; i < NL; ++i) g[i] = load16_any(base, off[i]);
  }
  // The same for a K step of which only the first kleft k exist (1 <= kleft < BK; KC: the row has at least CE
  // elements up to its end): chunks are moved back to end with the row (KC), rows of k past the end repeat the
  // last (MC).
  __device__ __forceinline__ void load_tail(const char* base, int64_t ld, int kleft, u32x4 (&g)[NL]) const {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      if constexpr (MC) {
        const int over = max(lrow + i * RPL - (kleft - 1), 0);
        g[i] = load16_any(base - (int64_t)over * ld * EB, off[i]);
      } else {
        const int over = max(element(i) + CE - kleft, 0);
        g[i] = load16_any(base - over * EB, off[i]);
      }
    }
  }
  __device__ __forceinline__ void fix_tail(int kleft, u32x4 (&g)[NL]) const {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      if constexpr (MC) {
        if (lrow + i * RPL >= kleft) g[i] = u32x4{0u, 0u, 0u, 0u};
      } else {
        g[i] = shift_bytes(g[i], max(element(i) + CE - kleft, 0) * EB);
      }
    }
  }
  // edge: some column of the tile does not exist (uniform).
  __device__ __forceinline__ void store(char* tile, int tid, bool edge, u32x4 (&g)[NL]) const {
    if constexpr (MC) {
      if (edge) {
#pragma unroll
        for (int i = 0; i < NL; ++i) g[i] = shift_bytes(g[i], shift);
      }
    }
#pragma unroll
    for (int i = 0; i < NL; ++i) *reinterpret_cast<u32x4*>(tile + (i * NT + tid) * 16) = g[i];
  }
};

// Fragments of a tile as AnyLoader lays it out: slab t of 32 rows, quarter ks of the K step.
//   16-bit: lane l holds row l % 32, k = 16 ks + 8 (l / 32) .. +7: one matrix instruction.
//   fp32: row l % 32, k = 8 ks + 4 (l / 32) .. +3: element j of both operands goes to the j-th of four 32x32x2
//         instructions (k = j and 4 + j of the eight, the same permutation for both operands).
template <typename T, bool MC, int ROWS, int TT>
struct AnyFrag {
  typedef typename Elem<T>::vec8 V;
  FragAddr<MC, ROWS, 64, TT> addr;
  __device__ __forceinline__ void init(int row0, int lane) { addr.init(row0, lane); }
  __device__ __forceinline__ V read(const char* tile, int t, int ks) const { return addr.template read<V>(tile, t, ks); }
};
template <bool MC, int ROWS, int TT>
struct AnyFrag<float, MC, ROWS, TT> {
  typedef floatx4 V;
  int base[MC ? 1 : 4];
  __device__ __forceinline__ void init(int row0, int lane) {
    const int row = row0 + (lane & 31), g = lane >> 5;
    if constexpr (MC) {
      base[0] = (4 * g * ROWS + row) * 4;
    } else {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) base[ks] = row * 128 + (((2 * ks + g) ^ swz<false, ROWS, 64>(row)) << 4);
    }
  }
  __device__ __forceinline__ V read(const char* tile, int t, int ks) const {
    if constexpr (MC) {
      V v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = *reinterpret_cast<const float*>(tile + base[0] + (8 * ks + j) * ROWS * 4 + t * 128);
      return v;
    } else {
      return *reinterpret_cast<const floatx4*>(tile + base[ks] + t * 4096);
    }
  }
};

// acc[i][j] += the products of fragments fb[j] and fa[i] (operands swapped: gemm_kernel.h).
template <typename T, int TM, int TN, typename V>
__device__ __forceinline__ void mma_block(floatx16 (&acc)[TM][TN], const V (&fa)[TM], const V (&fb)[TN]) {
  constexpr int J = sizeof(T) == 4 ? 4 : 1;
#pragma unroll
  for (int q = 0; q < J; ++q)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int jj = (i & 1) ? TN - 1 - j : j;  // boustrophedon: consecutive instructions share one operand
        if constexpr (sizeof(T) == 4) acc[i][jj] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[jj][q], fa[i][q], acc[i][jj], 0, 0, 0);
        else acc[i][jj] = Elem<T>::mfma(fb[jj], fa[i], acc[i][jj]);
      }
}

}  // namespace gemm_impl
