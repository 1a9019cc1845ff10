// MFMA GEMM for operands of any alignment: 16-bit ones whose rows do not start on 16-byte boundaries or do not
// hold whole 16-byte chunks (odd leading dimensions, odd K or N; the direct-to-LDS loads of gemm_kernel.h cannot
// take them), and fp32 ones on the small tile (on the large one: gemm_split.h, which comes here for what it cannot take).
//
// What bounds it: 16-bit, the load path (gemm_loader.h); fp32, the matrix instructions (256 flop per cycle and CU).
// A K step's chunks are loaded one or two whole steps before they are written to LDS, so that two LDS stages suffice
// and two work-groups of the large tile share a CU.
// Measured, microseconds (element-wise gathers -> here): bf16 1023 x 5003 x 2047 421 -> 56 (52 on operands that stay in
// the caches), 496 x 1331 x 13447 2930 -> 73, with scratch for a K split 59, 4001 x 4001 x 4001 189; fp32
// 2048 x 2048 x 1024 123 -> 71 on the large tile (121 TFLOP/s).
#pragma once
#include "gemm_loader.h"

namespace gemm_impl {

// Every wave's LDS stores are done and its reads have returned (global loads stay in flight).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

constexpr int ragged_lds_bytes(int bt) { return 4 * bt * 128; }

// The products of a BT x BT tile at (m0, n0): 2 x WGN waves, K step of 128 bytes, two LDS stages.
// acc[i][j][e] is out[m][n], m = m0 + 32 TM wm + 32 i + lane % 32, n = n0 + 32 TN wn + 32 j + 8 (e / 4) + 4 (lane / 32) + e % 4.
template <typename T, bool A_MC, bool B_MC, int BT, int WGN, bool MIS>
__device__ __forceinline__ void ragged_products(const typename AnyType<T>::Params& p, int m0, int n0, int64_t bz, int tid, char* lds,
                                                floatx16 (&acc)[BT / 64][BT / WGN / 32]) {
  constexpr int BK = 128 / sizeof(T), KS = AnyType<T>::KS;
  constexpr int NT = 2 * WGN * 64, TM = BT / 64, TN = BT / WGN / 32;
  constexpr int OP_BYTES = BT * 128, STAGE = 2 * OP_BYTES;
  static_assert(ragged_lds_bytes(BT) == 2 * STAGE, "two stages");
  typedef typename Elem<T>::vec8 V8;
  typedef AnyLoader<T, A_MC, BT, NT, MIS> LoaderA;
  typedef AnyLoader<T, B_MC, BT, NT, MIS> LoaderB;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;
  const int64_t k0 = bz * p.kslice;  // K slices (kslice > 0): grid member z takes k0 .. k0 + kslice - 1
  const int K = p.kslice ? min(p.K - (int)k0, p.kslice) : p.K;
  LoaderA la;
  LoaderB lb;
  la.init(reinterpret_cast<const T*>(p.a) + bz * p.sa, p.lda, m0, p.M, k0, p.K, tid);
  lb.init(reinterpret_cast<const T*>(p.b) + bz * p.sb, p.ldb, n0, p.N, k0, p.K, tid);

#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = zero16();

  const int KT = (K + BK - 1) / BK;
  struct Regs {
    typename LoaderA::Regs a;
    typename LoaderB::Regs b;
  };
  // Chunks on their way: of the even and of the odd K steps, or of one step only (fp32, whose large tile's step is
  // longer than a load takes).
  constexpr bool TWO = BT == 64 || MIS;
  Regs even, odd;
  auto load = [&](Regs& g) {
    la.load(g.a);
    lb.load(g.b);
  };
  auto store = [&](Regs& g, char* stage) {
    la.store(stage, g.a);
    lb.store(stage + OP_BYTES, g.b);
  };
  load(even);
  if (TWO && KT > 1) load(odd);
  store(even, lds);
  if (KT > (TWO ? 2 : 1)) load(even);
  lds_barrier();

  AnyFrag<T, A_MC, BT, TM> faddr;
  AnyFrag<T, B_MC, BT, TN> fbddr;
  faddr.init(wm * 32 * TM, lane);
  fbddr.init(wn * 32 * TN, lane);
  V8 fa[2][TM], fb[2][TN];
  auto read_frags = [&](const char* stage, int ks, int buf) {
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[buf][i] = faddr.read(stage, i, ks);
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[buf][j] = fbddr.read(stage + OP_BYTES, j, ks);
  };
  // K step kt, with step kt + 1 in the registers g: those go to LDS, and another step is sent for.
  auto step = [&](int kt, Regs& g, const char* cur, char* nxt) {
    store(g, nxt);
    if (kt + (TWO ? 3 : 2) < KT) load(g);
    __builtin_amdgcn_sched_barrier(0);  // (the loads would sink behind the matrix instructions)
    static_for<KS>([&](auto KSI) {
      constexpr int ks = decltype(KSI)::value;
      if constexpr (ks + 1 < KS) {
        read_frags(cur, ks + 1, (ks + 1) & 1);
      } else {
        lds_barrier();
        read_frags(nxt, 0, KS & 1);
      }
      mma_block<T, TM, TN>(acc, fa[ks & 1], fb[ks & 1]);
    });
  };
  read_frags(lds, 0, 0);
  int kt = 0;
  for (; kt + 2 < KT; kt += 2) {
    step(kt, TWO ? odd : even, lds, lds + STAGE);
    step(kt + 1, even, lds + STAGE, lds);
  }
  if (kt + 1 < KT) step(kt++, TWO ? odd : even, lds, lds + STAGE);
  // The last K step, of which only some k may exist.
  const int tail = K - kt * BK;
  const char* last = lds + (kt & 1) * STAGE;
  static_for<KS>([&](auto KSI) {
    constexpr int ks = decltype(KSI)::value;
    if constexpr (ks + 1 < KS) read_frags(last, ks + 1, (ks + 1) & 1);
#pragma unroll
    for (int i = 0; i < TM; ++i) mask_fragment<T>(fa[ks & 1][i], ks, lane, tail);
#pragma unroll
    for (int j = 0; j < TN; ++j) mask_fragment<T>(fb[ks & 1][j], ks, lane, tail);
    mma_block<T, TM, TN>(acc, fa[ks & 1], fb[ks & 1]);
  });
}

// The same tile as a kernel of its own.
template <typename T, bool OutF32, bool A_MC, bool B_MC, int BT, int WGN, bool MIS>
__global__ __launch_bounds__(2 * WGN * 64) void gemm_ragged_kernel(typename AnyType<T>::Params p) {
  constexpr int TM = BT / 64, TN = BT / WGN / 32;
  __shared__ __attribute__((aligned(1024))) char lds[ragged_lds_bytes(BT)];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;

  request_first_args(p);
  const TileAt tile = tile_at(blockIdx.x, p.order);
  const int m0 = tile.m * BT, n0 = tile.n * BT;
  const int64_t bz = blockIdx.z;
  floatx16 acc[TM][TN];
  ragged_products<T, A_MC, B_MC, BT, WGN, MIS>(p, m0, n0, bz, tid, lds, acc);

  lds_barrier();  // every wave has read its last fragments
  typename AnyType<T>::template Epilogue<OutF32> epi(p, bz);
  store_tile<typename AnyType<T>::Out, OutF32>(epi, acc, lds + wave * (TN * 4096), member_out(p, bz), p.ldc, bz * p.sc, p.M, p.N, m0 + wm * 32 * TM,
                        n0 + wn * 32 * TN, lane);
}

template <typename T, bool OutF32, bool A_MC, bool B_MC>
void launch_ragged_tile(typename AnyType<T>::Params& p, int batch, int tile, hipStream_t st) {
  p.tiles_m = (int)xmk::ceil_div(p.M, tile);
  p.tiles_n = (int)xmk::ceil_div(p.N, tile);
  p.order = tile_order((uint32_t)p.tiles_m, (uint32_t)p.tiles_n, p.K);
  const dim3 grid((unsigned)(p.tiles_m * p.tiles_n), 1, (unsigned)batch);
  if constexpr (sizeof(T) != 2) {  // (16-bit operands without misaligned rows take the direct kernels)
    if (!p.misaligned) {
      if (tile == 128) hipLaunchKernelGGL((gemm_ragged_kernel<T, OutF32, A_MC, B_MC, 128, 2, false>), grid, dim3(256), 0, st, p);
      else hipLaunchKernelGGL((gemm_ragged_kernel<T, OutF32, A_MC, B_MC, 64, 2, false>), grid, dim3(256), 0, st, p);
      return;
    }
  }
  if (tile == 128) hipLaunchKernelGGL((gemm_ragged_kernel<T, OutF32, A_MC, B_MC, 128, 2, true>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((gemm_ragged_kernel<T, OutF32, A_MC, B_MC, 64, 2, true>), grid, dim3(256), 0, st, p);
}

template <typename T, bool OutF32>
void launch_ragged_impl(bool a_mc, bool b_mc, typename AnyType<T>::Params& p, int batch, int tile, hipStream_t st) {
  if (!a_mc && !b_mc) launch_ragged_tile<T, OutF32, false, false>(p, batch, tile, st);
  else if (!a_mc && b_mc) launch_ragged_tile<T, OutF32, false, true>(p, batch, tile, st);
  else if (a_mc && !b_mc) launch_ragged_tile<T, OutF32, true, false>(p, batch, tile, st);
  else launch_ragged_tile<T, OutF32, true, true>(p, batch, tile, st);
}

// Explicitly instantiated in gemm_inst_ragged_*.hip.
template <typename T, bool OutF32>
void launch_ragged(bool a_mc, bool b_mc, typename AnyType<T>::Params& p, int batch, int tile, hipStream_t st);

}  // namespace gemm_impl
