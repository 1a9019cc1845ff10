// Operand tiles for the kernels that take any alignment (gemm_ragged.h, gemm_slices.h): global memory -> registers
// -> LDS in 16-byte chunks, and the matrix-core fragments read back from LDS.
//
// A K step is 128 bytes of a reduction-contiguous row: 64 elements of 16 bits, 32 of fp32, 128 of fp8.
//   KC operand (reduction index contiguous): LDS [row][128 bytes], chunks XORed by pairs of rows.
//   MC operand (free index contiguous): LDS [k][rows], 8- and 16-bit elements read with the transpose loads, fp32
//       ones as scalars.
// Rows may start on any element: every lane fetches whole chunks, at whatever byte address they lie (the hardware
// takes global loads at any), never element by element.  Nothing branches and nothing outside the operand is read:
// a chunk that would reach past the operand's end is read from 16 bytes before it and shifted into place, and what
// lies past the end of K is masked in the last step's fragments.
// At an unaligned address the address unit takes the 64 lanes of a load one by one (64 cycles of the CU's load path
// instead of 16; by the cache-access counter 58 accesses per load: 75 thousand cycles of each CU's path in the 124 thousand
// of 1023 x 5003 x 2047, whose waves wait 45 % of their time for an instruction to issue), which bounds the large products.
// Loading the aligned chunks around it instead and picking each lane's piece out of its own and its neighbour's (24 vector
// instructions per chunk) was level there and slower on 4001^3 (191 -> 224 us) and on the slices kernel: the vector issue
// port then is what the address unit was.
#pragma once
#include "gemm_kernel.h"

namespace gemm_impl {

// What the kernels need to know of an element type beyond Elem: the kernel's parameters, the type of 16-bit results,
// the fragments of a K step, and the epilogue.
template <typename T> struct AnyType {
  typedef GemmParams Params;
  typedef T Out;
  static constexpr int KS = 4;
  template <bool OutF32> using Epilogue = GemmEpilogue<T, OutF32>;
};

template <> struct Elem<float> {
  typedef floatx4 vec8;  // four consecutive k: operands of four matrix instructions
  static __device__ __forceinline__ float to_f32(float v) { return v; }
  static __device__ __forceinline__ uint16_t from_f32(float) { return 0; }  // fp32 outputs only
};

// v moved down by `bytes` (>= 0), zeros behind.
__device__ __forceinline__ u32x4 shift_bytes(u32x4 v, uint32_t bytes) {
  const uint32_t d = bytes >> 2;
  if (d & 1) v = u32x4{v[1], v[2], v[3], 0u};
  if (d & 2) v = u32x4{v[2], v[3], 0u, 0u};
  if (d & ~3u) v = u32x4{0u, 0u, 0u, 0u};
  const uint32_t b = bytes & 3;
  return u32x4{__builtin_amdgcn_alignbyte(v[1], v[0], b), __builtin_amdgcn_alignbyte(v[2], v[1], b),
               __builtin_amdgcn_alignbyte(v[3], v[2], b), __builtin_amdgcn_alignbyte(0u, v[3], b)};
}

// One operand tile of ROWS rows (or columns) x one K step, fetched by NT threads as NL chunks of 16 bytes each.
// Thread t takes chunk t % CPR of the LDS rows t / CPR + i RPL.
// MIS: rows may start anywhere; otherwise every row starts on a 16-byte boundary (its length may be anything; the
// chunk with an operand's last bytes then ends inside the 16-byte granule that holds them).
template <typename T, bool MC, int ROWS, int NT, bool MIS>
struct AnyLoader {
  static constexpr int EB = sizeof(T), BK = 128 / EB;
  static constexpr int RB = MC ? ROWS * EB : 128;  // bytes of an LDS row
  static constexpr int CPR = RB / 16;              // chunks per LDS row
  static constexpr int RPL = NT / CPR;             // LDS rows per load
  static constexpr int NL = ROWS * 8 / NT;
  static_assert(NL >= 1 && RPL % (EB == 1 ? 8 : 4) == 0 && (MC || RPL % 8 == 0), "the swizzle repeats, or changes by store()'s term");
  struct Regs {
    u32x4 g[NL];
    int32_t limit;  // (uniform) the largest offset that could be loaded from
  };
  const char* base;    // the next K step's origin
  int64_t left, step;  // from there to the last place a chunk can be loaded from; to the next K step
  uint32_t off[NL];    // byte offsets of the lane's chunks
  int32_t reach;       // (uniform) no lane's offset is larger
  int lds0;            // LDS byte offset of chunk 0

  static __device__ __forceinline__ int swizzle(int row_or_k) {
    if constexpr (MC && EB == 4) return 0;
    // 8-bit transpose reads: 32 lanes take 32 bytes of each of 8 consecutive k
    else if constexpr (MC && EB == 1) return ROWS < 64 ? 0 : ROWS < 128 ? ((row_or_k >> 2) & 1) << 1 : ((row_or_k >> 1) & 3) << 1;
    else return swz<MC, ROWS, 64>(row_or_k);
  }
  // op: the operand (of this batch member), rows x depth elements (stored depth x rows when MC), ld elements from one
  // stored row to the next; at least 16 bytes in all.  The tile starts at row (column) row0 and at reduction index k0.
  __device__ __forceinline__ void init(const T* op, int64_t ld, int row0, int rows, int64_t k0, int depth, int tid) {
    const T* origin = op + (MC ? k0 * ld + row0 : (int64_t)row0 * ld + k0);
    const T* past = op + (MC ? (int64_t)(depth - 1) * ld + rows : (int64_t)(rows - 1) * ld + depth);
    base = reinterpret_cast<const char*>(origin);
    left = (reinterpret_cast<const char*>(past) - base) - 16;
    if constexpr (!MIS) left = (left + 15) & ~(int64_t)15;
    step = MC ? BK * ld * EB : 128;
    const int lrow = tid / CPR, c = tid % CPR;
    lds0 = lrow * RB + ((c ^ swizzle(lrow)) << 4);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      int r = lrow + i * RPL;
      if constexpr (!MC) r = min(r, rows - 1 - row0);  // rows past the end repeat the last one: their products are not stored
      off[i] = (uint32_t)((int64_t)r * ld * EB) + c * 16;
    }
    const int r = MC ? BK - 1 : min(ROWS, rows - row0) - 1;
    reach = (int32_t)((int64_t)r * ld * EB) + RB - 16;
  }
  __device__ __forceinline__ void advance(int steps) {
    base += steps * step;
    left -= steps * step;
  }
  // Sends for the next K step.
  __device__ __forceinline__ void load(Regs& r) {
    r.limit = (int32_t)min(left, (int64_t)0x7ffffff0);
    const char* from = r.limit < 0 ? base + r.limit : base;
    const uint32_t cap = (uint32_t)max(r.limit, 0);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const uint32_t at = min(off[i], cap);
      if constexpr (MIS) __builtin_memcpy(&r.g[i], from + at, 16);
      else r.g[i] = *reinterpret_cast<const u32x4*>(from + at);
    }
    advance(1);
  }
  // Moves what was read from before an operand's end into place.
  __device__ __forceinline__ void shift_ends(Regs& r) const {
    if constexpr (MIS) {
      if (reach > r.limit) {  // only at the operand's end
#pragma unroll
        for (int i = 0; i < NL; ++i) r.g[i] = shift_bytes(r.g[i], (uint32_t)max((int32_t)off[i] - r.limit, 0));
      }
    }
  }
  __device__ __forceinline__ void store(char* tile, Regs& r) const {
    shift_ends(r);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      // (KC: the XOR counts pairs of rows modulo 16 rows)
      const int at = (!MC && RPL % 16 != 0 && (i & 1)) ? lds0 ^ 64 : lds0;
      *reinterpret_cast<u32x4*>(tile + at + i * RPL * RB) = r.g[i];
    }
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

// Zeroes the elements of a fragment (quarter ks of a K step) from k = kleft on.
template <typename T, typename V>
__device__ __forceinline__ void mask_fragment(V& v, int ks, int lane, int kleft) {
  if constexpr (sizeof(T) == 1) {
    const int n = kleft - (2 * ks + (lane >> 5)) * 32;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int b = min(max(n - 4 * q, 0), 4);  // bytes of the word that exist
      v[q] &= b == 4 ? -1 : (1 << (8 * b)) - 1;
    }
    return;
  } else {
  constexpr int E = sizeof(T) == 4 ? 4 : 8;  // consecutive k of a lane
  const int n = kleft - (2 * ks + (lane >> 5)) * E;
  u32x4 w = __builtin_bit_cast(u32x4, v);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if constexpr (E == 4) w[q] = n > q ? w[q] : 0u;
    else w[q] &= n >= 2 * q + 2 ? 0xffffffffu : n == 2 * q + 1 ? 0xffffu : 0u;
  }
  v = __builtin_bit_cast(V, w);
  }
}

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
