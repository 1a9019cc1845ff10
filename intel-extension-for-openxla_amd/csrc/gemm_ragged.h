// MFMA GEMM for operands of any alignment: 16-bit ones whose rows do not start on 16-byte boundaries or do not
// hold whole 16-byte chunks (odd leading dimensions, odd K or N; the direct-to-LDS loads of gemm_kernel.h cannot
// take them), and all fp32 ones.
//
// What bounds it: 16-bit, the load path (rows start on any 2-byte boundary, so a 128-byte row segment touches two
// cache lines, and the data passes through registers); fp32, the matrix instructions (256 flop per cycle and CU).
// A K step's chunks are loaded one whole step before they are written to LDS, so that two LDS stages suffice and
// two work-groups of the large tile share a CU.
// Measured, bf16, microseconds (element-wise gathers -> here): 1023 x 5003 x 2047 421 -> 57, 496 x 1331 x 13447
// 2930 -> 106, 63 x 63 x 1023 95 -> 8.8 (64 x 64 x 1024 on the direct kernel: 7.1).
#pragma once
#include "gemm_loader.h"

namespace gemm_impl {

// BT x BT tile, 256 threads = 4 waves in 2 x 2, K step of 128 bytes, two LDS stages.
template <typename T, bool OutF32, bool A_MC, bool B_MC, int BT>
__global__ __launch_bounds__(256) void gemm_ragged_kernel(GemmParams p) {
  constexpr int BK = 128 / sizeof(T), KS = 4;
  constexpr int WT = BT / 2, TT = WT / 32;
  constexpr int OP_BYTES = BT * 128, STAGE = 2 * OP_BYTES;
  typedef typename Elem<T>::vec8 V8;
  typedef AnyLoader<T, A_MC, BT, 256> LoaderA;
  typedef AnyLoader<T, B_MC, BT, 256> LoaderB;
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
  const int64_t a_step = (A_MC ? BK * p.lda : BK) * (int64_t)sizeof(T), b_step = (B_MC ? BK * p.ldb : BK) * (int64_t)sizeof(T);
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

  AnyFrag<T, A_MC, BT, TT> faddr;
  AnyFrag<T, B_MC, BT, TT> fbddr;
  faddr.init(wm * WT, lane);
  fbddr.init(wn * WT, lane);
  V8 fa[2][TT], fb[2][TT];
  auto read_frags = [&](const char* stage, int ks, int buf) {
#pragma unroll
    for (int i = 0; i < TT; ++i) fa[buf][i] = faddr.read(stage, i, ks);
#pragma unroll
    for (int j = 0; j < TT; ++j) fb[buf][j] = fbddr.read(stage + OP_BYTES, j, ks);
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
      mma_block<T, TT, TT>(acc, fa[ks & 1], fb[ks & 1]);
    });
  }

  // acc[i][j][e] is out[m][n], m = m0 + wm WT + 32 i + lane % 32, n = n0 + wn WT + 32 j + 8 (e / 4) + 4 (lane / 32) + e % 4.
  barrier();  // every wave has read its last fragments
  GemmEpilogue<T, OutF32> epi(p, bz);
  store_tile<T, OutF32>(epi, acc, lds + wave * (TT * 4096), member_out(p, bz), p.ldc, bz * p.sc, p.M, p.N, m0 + wm * WT, n0 + wn * WT, lane);
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
