// 16-bit MFMA GEMM for operands whose rows do not start on 16-byte boundaries or do not hold whole 16-byte
// chunks (odd leading dimensions, odd K or N): the operands that the direct-to-LDS loads of gemm_kernel.h
// cannot take.
//
// What bounds it: the load path.  Rows start on any 2-byte boundary, so a 128-byte row segment touches two
// cache lines, and the data must pass through registers.  Every lane still fetches whole 16-byte chunks (the
// hardware takes global loads at any byte address), never element by element: a chunk that would reach past the
// end of its row is read from 16 bytes before that end and shifted into place, so nothing outside the matrix
// is touched and no lane branches.  A K step's chunks are loaded one whole step before they are written to LDS,
// so that two LDS stages suffice and two work-groups of the large tile share a CU.
// LDS layouts, fragments and the MFMA order are those of gemm_kernel.h.
// Measured, bf16, microseconds (element-wise gathers -> here): 1023 x 5003 x 2047 421 -> 57, 496 x 1331 x 13447
// 2930 -> 106, 63 x 63 x 1023 95 -> 8.8 (64 x 64 x 1024 on the direct kernel: 7.1).
#pragma once
#include "gemm_kernel.h"

namespace gemm_impl {

// v shifted towards element 0 by s 16-bit elements, zeros behind (s >= 8: all zero).
__device__ __forceinline__ u32x4 shift_elements(u32x4 v, int s) {
  const int d = s >> 1;
  if (d & 1) v = u32x4{v[1], v[2], v[3], 0u};
  if (d & 2) v = u32x4{v[2], v[3], 0u, 0u};
  if (d & ~3) v = u32x4{0u, 0u, 0u, 0u};
  if (s & 1) v = u32x4{__builtin_amdgcn_alignbit(v[1], v[0], 16), __builtin_amdgcn_alignbit(v[2], v[1], 16),
                       __builtin_amdgcn_alignbit(v[3], v[2], 16), v[3] >> 16};
  return v;
}

__device__ __forceinline__ u32x4 load16_any(const char* base, uint32_t off) {
  u32x4 v;
  __builtin_memcpy(&v, base + off, 16);  // one global_load_dwordx4 at any alignment
  return v;
}

// One operand tile of ROWS rows (or columns) x BK k, fetched by NT threads as NL chunks of 16 bytes each.
// Chunk i of thread t goes to LDS bytes [16 (i NT + t), +16).
template <bool MC, int ROWS, int BK, int NT>
struct RaggedLoader {
  static constexpr int RB = MC ? ROWS * 2 : BK * 2;
  static constexpr int CPR = RB / 16;
  static constexpr int RPL = NT / CPR;  // LDS rows per load
  static constexpr int NL = ROWS * BK * 2 / 16 / NT;
  static_assert(NL >= 1 && RPL % 8 == 0, "the swizzle repeats from load to load");
  uint32_t off[NL];  // byte offset of chunk i from the operand's K step origin
  int lrow, c0;      // LDS row of chunk 0; first element of the chunks within their LDS row
  int shift;         // MC: elements by which the chunks were moved back to stay inside their rows

  // row0: first row (KC) or column (MC) of the tile; rows: how many the matrix has.
  __device__ __forceinline__ void init(int64_t ld, int row0, int rows, int tid) {
    lrow = tid / CPR;
    c0 = ((tid % CPR) ^ swz<MC, ROWS, BK>(lrow)) * 8;
    shift = 0;
    if constexpr (MC) {
      const int col = row0 + c0, at = min(col, rows - 8);  // rows >= 8
      shift = col - at;
#pragma unroll
      for (int i = 0; i < NL; ++i) off[i] = (uint32_t)(((int64_t)(lrow + i * RPL) * ld + at) * 2);
    } else {
#pragma unroll
      for (int i = 0; i < NL; ++i) {  // rows past the end repeat the last one: their products are not stored
        const int r = min(row0 + lrow + i * RPL, rows - 1) - row0;
        off[i] = (uint32_t)(((int64_t)r * ld + c0) * 2);
      }
    }
  }
  // base: the operand at this K step's first k (KC: of the tile's first row).
  __device__ __forceinline__ void load(const char* base, u32x4 (&g)[NL]) const {
#pragma unroll
    for (int i = 0; i < NL; ++i) g[i] = load16_any(base, off[i]);
  }
  // The same for a K step of which only the first kleft k exist (1 <= kleft < BK; the row has at least 8 elements
  // up to its end): chunks are moved back to end with the row (KC), rows of k past the end repeat the last (MC).
  __device__ __forceinline__ void load_tail(const char* base, int64_t ld, int kleft, u32x4 (&g)[NL]) const {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      if constexpr (MC) {
        const int over = max(lrow + i * RPL - (kleft - 1), 0);
        g[i] = load16_any(base - (int64_t)over * ld * 2, off[i]);
      } else {
        const int over = max(c0 + 8 - kleft, 0);
        g[i] = load16_any(base - over * 2, off[i]);
      }
    }
  }
  __device__ __forceinline__ void fix_tail(int kleft, u32x4 (&g)[NL]) const {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      if constexpr (MC) {
        if (lrow + i * RPL >= kleft) g[i] = u32x4{0u, 0u, 0u, 0u};
      } else {
        g[i] = shift_elements(g[i], max(c0 + 8 - kleft, 0));
      }
    }
  }
  // edge: some column of the tile does not exist (uniform over the work-group).
  __device__ __forceinline__ void store(char* tile, int tid, bool edge, u32x4 (&g)[NL]) const {
    if constexpr (MC) {
      if (edge) {
#pragma unroll
        for (int i = 0; i < NL; ++i) g[i] = shift_elements(g[i], shift);
      }
    }
#pragma unroll
    for (int i = 0; i < NL; ++i) *reinterpret_cast<u32x4*>(tile + (i * NT + tid) * 16) = g[i];
  }
};

// BT x BT tile, 256 threads = 4 waves in 2 x 2, K step 64, two LDS stages.
template <typename T, bool OutF32, bool A_MC, bool B_MC, int BT>
__global__ __launch_bounds__(256) void gemm_ragged_kernel(GemmParams p) {
  constexpr int BK = 64, KS = BK / 16;
  constexpr int WT = BT / 2, TT = WT / 32;
  constexpr int OP_BYTES = BT * BK * 2, STAGE = 2 * OP_BYTES;
  typedef typename Elem<T>::vec8 V8;
  typedef RaggedLoader<A_MC, BT, BK, 256> LoaderA;
  typedef RaggedLoader<B_MC, BT, BK, 256> LoaderB;
  __shared__ __attribute__((aligned(1024))) char lds[2 * STAGE];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  int pid = blockIdx.x;  // tile order: as in gemm_mfma_kernel
  const int ntiles = p.tiles_m * p.tiles_n;
  if (ntiles % 8 == 0) pid = (pid % 8) * (ntiles / 8) + pid / 8;
  constexpr int GM = 8;
  const int group = pid / (GM * p.tiles_n);
  const int first_m = group * GM;
  const int gsize = min(p.tiles_m - first_m, GM);
  const int m0 = (first_m + (pid % (GM * p.tiles_n)) % gsize) * BT;
  const int n0 = (pid % (GM * p.tiles_n)) / gsize * BT;

  const int64_t bz = blockIdx.z;
  const int64_t k0 = bz * p.kslice;  // K slices (kslice > 0): grid member z takes k0 .. k0 + kslice - 1
  const int K = p.kslice ? min(p.K - (int)k0, p.kslice) : p.K;
  // MC operands are addressed from column 0 (a chunk may start before the tile's first column).
  const char* a_base = (const char*)(reinterpret_cast<const T*>(p.a) + bz * p.sa + (A_MC ? k0 * p.lda : (int64_t)m0 * p.lda + k0));
  const char* b_base = (const char*)(reinterpret_cast<const T*>(p.b) + bz * p.sb + (B_MC ? k0 * p.ldb : (int64_t)n0 * p.ldb + k0));
  const int64_t a_step = (A_MC ? BK * p.lda : BK) * 2, b_step = (B_MC ? BK * p.ldb : BK) * 2;
  const bool a_edge = A_MC && m0 + BT > p.M, b_edge = B_MC && n0 + BT > p.N;
  LoaderA la;
  LoaderB lb;
  la.init(p.lda, m0, p.M, tid);
  lb.init(p.ldb, n0, p.N, tid);

  floatx16 acc[TT][TT];
#pragma unroll
  for (int i = 0; i < TT; ++i)
#pragma unroll
    for (int j = 0; j < TT; ++j) acc[i][j] = zero16();

  const int KT = (K + BK - 1) / BK;
  u32x4 ga[LoaderA::NL], gb[LoaderB::NL];
  auto load = [&](int kt) {
    const int kleft = K - kt * BK;
    if (kleft >= BK) {
      la.load(a_base, ga);
      lb.load(b_base, gb);
    } else {
      la.load_tail(a_base, p.lda, kleft, ga);
      lb.load_tail(b_base, p.ldb, kleft, gb);
    }
    a_base += a_step;
    b_base += b_step;
  };
  auto store = [&](int kt, char* stage) {
    const int kleft = K - kt * BK;
    if (kleft < BK) {
      la.fix_tail(kleft, ga);
      lb.fix_tail(kleft, gb);
    }
    la.store(stage, tid, a_edge, ga);
    lb.store(stage + OP_BYTES, tid, b_edge, gb);
  };
  // Every wave's LDS stores are done and its reads have returned (global loads stay in flight).
  auto barrier = [&] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  load(0);
  store(0, lds);
  if (KT > 1) load(1);
  barrier();

  FragAddr<A_MC, BT, BK, TT> faddr;
  FragAddr<B_MC, BT, BK, TT> fbddr;
  faddr.init(wm * WT, lane);
  fbddr.init(wn * WT, lane);
  V8 fa[2][TT], fb[2][TT];
  auto read_frags = [&](const char* stage, int ks, int buf) {
#pragma unroll
    for (int i = 0; i < TT; ++i) fa[buf][i] = faddr.template read<V8>(stage, i, ks);
#pragma unroll
    for (int j = 0; j < TT; ++j) fb[buf][j] = fbddr.template read<V8>(stage + OP_BYTES, j, ks);
  };
  read_frags(lds, 0, 0);
  for (int kt = 0; kt < KT; ++kt) {
    char* cur = lds + (kt & 1) * STAGE;
    char* nxt = lds + ((kt + 1) & 1) * STAGE;
    if (kt + 1 < KT) store(kt + 1, nxt);
    if (kt + 2 < KT) load(kt + 2);
    static_for<KS>([&](auto KSI) {
      constexpr int ks = decltype(KSI)::value;
      if constexpr (ks + 1 < KS) {
        read_frags(cur, ks + 1, (ks + 1) & 1);
      } else if (kt + 1 < KT) {
        barrier();
        read_frags(nxt, 0, KS & 1);
      }
#pragma unroll
      for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int j = 0; j < TT; ++j) {
          const int jj = (i & 1) ? TT - 1 - j : j;
          acc[i][jj] = Elem<T>::mfma(fb[ks & 1][jj], fa[ks & 1][i], acc[i][jj]);
        }
    });
  }

  // acc[i][j][e] is out[m][n], m = m0 + wm WT + 32 i + lane % 32, n = n0 + wn WT + 32 j + 8 (e / 4) + 4 (lane / 32) + e % 4.
  barrier();  // every wave has read its last fragments
  GemmEpilogue<T, OutF32> epi(p, bz);
  store_tile<T, OutF32>(epi, acc, lds + wave * (TT * 4096), member_out(p, bz), p.ldc, bz * p.sc, p.M, p.N, m0 + wm * WT, n0 + wn * WT, lane);
}

// Tile edge of the ragged kernel: 128 where such tiles keep most CUs busy, else 64.
constexpr int kRaggedTiles128 = 160;
inline int ragged_tile(int64_t m, int64_t n, int64_t batch) {
  return xmk::ceil_div(m, 128) * xmk::ceil_div(n, 128) * batch >= kRaggedTiles128 ? 128 : 64;
}

template <typename T, bool OutF32, bool A_MC, bool B_MC>
void launch_ragged_tile(GemmParams& p, int batch, int tile, hipStream_t st) {
  p.tiles_m = (int)xmk::ceil_div(p.M, tile);
  p.tiles_n = (int)xmk::ceil_div(p.N, tile);
  const dim3 grid((unsigned)(p.tiles_m * p.tiles_n), 1, (unsigned)batch);
  if (tile == 128) hipLaunchKernelGGL((gemm_ragged_kernel<T, OutF32, A_MC, B_MC, 128>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((gemm_ragged_kernel<T, OutF32, A_MC, B_MC, 64>), grid, dim3(256), 0, st, p);
}

template <typename T, bool OutF32>
void launch_ragged_impl(bool a_mc, bool b_mc, GemmParams& p, int batch, int tile, hipStream_t st) {
  if (!a_mc && !b_mc) launch_ragged_tile<T, OutF32, false, false>(p, batch, tile, st);
  else if (!a_mc && b_mc) launch_ragged_tile<T, OutF32, false, true>(p, batch, tile, st);
  else if (a_mc && !b_mc) launch_ragged_tile<T, OutF32, true, false>(p, batch, tile, st);
  else launch_ragged_tile<T, OutF32, true, true>(p, batch, tile, st);
}

// Explicitly instantiated in gemm_inst_ragged_*.hip.
template <typename T, bool OutF32>
void launch_ragged(bool a_mc, bool b_mc, GemmParams& p, int batch, int tile, hipStream_t st);

}  // namespace gemm_impl
