// MFMA GEMM for products with too few output tiles to fill the device: a small tile per work-group, the reduction
// split over the work-group's waves.
//
// What bounds these products is latency, not a rate: with one 64 x 64 tile per CU the tile kernels spend 0.3 us per
// 64 k waiting for the three K steps they keep in flight.  Here each of the NW waves owns the whole 32 TM x 32 TN
// tile for every NW-th K step, keeps one or two of its K steps in flight in registers (NW times the bytes in flight per
// CU), passes them through an LDS region of its own (no barrier in the loop: the LDS serves a wave in order), and
// the waves' partial sums meet in LDS once at the end, added in wave order.  Small tiles also make more
// work-groups out of a small output.  Operands of any alignment, 16-bit and fp32 (gemm_loader.h).
// Measured without a K split, microseconds, weights from memory, best tile kernel -> best of these: bf16 1 x 4096 x 16384
// 80.7 -> 34.0 (B stored [N, K]), 120 x 1832 x 7296 44.2 -> 24.3, 2 x 96 x 9856 30.0 -> 16.7; odd rows 37 x 3441 x 9089
// 83.7 -> 35.4; fp32 6 x 336 x 14592 306 -> 67.  By the counters (64 x 4096 x 1024, 6.1 us) the waves wait three quarters
// of their time, the matrix cores are busy 4 %.
#pragma once
#include "gemm_loader.h"

namespace gemm_impl {

template <typename T, bool OutF32, bool A_MC, bool B_MC, int TM, int TN, int NW, bool MIS>
__global__ __launch_bounds__(NW * 64) void gemm_slices_kernel(typename AnyType<T>::Params p) {
  constexpr int BK = 128 / sizeof(T), KS = AnyType<T>::KS;
  constexpr int STAGE = (TM + TN) * 4096;                 // LDS per wave
  constexpr int RBY = TN * 128, XM = TN == 1 ? 7 : 15;    // partial sums: as in store_tile
  static_assert(STAGE >= TM * TN * 4096, "a wave's partial sums replace its operands");
  typedef AnyLoader<T, A_MC, 32 * TM, 64, MIS> LoaderA;
  typedef AnyLoader<T, B_MC, 32 * TN, 64, MIS> LoaderB;
  typedef typename Elem<T>::vec8 V8;
  __shared__ __attribute__((aligned(1024))) char lds[NW * STAGE];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  request_first_args(p);
  const TileAt tile = tile_at(blockIdx.x, p.order);
  const int m0 = tile.m * (32 * TM), n0 = tile.n * (32 * TN);

  const int64_t bz = blockIdx.z;
  const int64_t k0 = bz * p.kslice;  // as in gemm_ragged_kernel
  const int K = p.kslice ? min(p.K - (int)k0, p.kslice) : p.K;
  LoaderA la;
  LoaderB lb;
  la.init(reinterpret_cast<const T*>(p.a) + bz * p.sa, p.lda, m0, p.M, k0, p.K, lane);
  lb.init(reinterpret_cast<const T*>(p.b) + bz * p.sb, p.ldb, n0, p.N, k0, p.K, lane);
  la.advance(wave);  // K step `wave`, and every NW-th from there
  lb.advance(wave);
  la.step *= NW;
  lb.step *= NW;
  AnyFrag<T, A_MC, 32 * TM, TM> faddr;
  AnyFrag<T, B_MC, 32 * TN, TN> fbddr;
  faddr.init(0, lane);
  fbddr.init(0, lane);

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = zero16();

  const int KT = (K + BK - 1) / BK;
  char* region = lds + wave * STAGE;
  struct Regs {
    typename LoaderA::Regs a;
    typename LoaderB::Regs b;
  };
  constexpr bool TWO = TM * TN < 4;  // K steps in flight per wave: two, or one where the registers allow no more
  Regs r0, r1;
  auto load = [&](Regs& r) {
    la.load(r.a);
    lb.load(r.b);
  };
  // Multiplies K step kt, which is in the registers r, and sends the next but one (or the next) of this wave into
  // them.  LAST: the wave's last step, of which only some k may exist.
  auto step = [&](auto LAST, int kt, Regs& r) {
    la.store(region, r.a);
    lb.store(region + TM * 4096, r.b);
    if constexpr (!decltype(LAST)::value) {
      if (!TWO || kt + 2 * NW < KT) load(r);
      __builtin_amdgcn_sched_barrier(0);  // (the loads would sink behind the matrix instructions)
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      V8 fa[TM], fb[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[i] = faddr.read(region, i, ks);
#pragma unroll
      for (int j = 0; j < TN; ++j) fb[j] = fbddr.read(region + TM * 4096, j, ks);
      if constexpr (decltype(LAST)::value) {
#pragma unroll
        for (int i = 0; i < TM; ++i) mask_fragment<T>(fa[i], ks, lane, K - kt * BK);
#pragma unroll
        for (int j = 0; j < TN; ++j) mask_fragment<T>(fb[j], ks, lane, K - kt * BK);
      }
      mma_block<T, TM, TN>(acc, fa, fb);
    }
  };
  constexpr std::false_type inner;
  constexpr std::true_type last;
  int kt = wave;
  if (kt < KT) load(r0);
  if (TWO && kt + NW < KT) load(r1);
  for (; kt + 2 * NW < KT; kt += 2 * NW) {
    step(inner, kt, r0);
    step(inner, kt + NW, TWO ? r1 : r0);
  }
  if (kt + NW < KT) {
    step(inner, kt, r0);
    step(last, kt + NW, TWO ? r1 : r0);
  } else if (kt < KT) {
    step(last, kt, r0);
  }

  // The waves' partial sums, in store_tile's layout (slab i of 32 rows after the other).
  const int row32 = lane & 31, h = lane >> 5;
  static_for<TM>([&](auto I) {
    constexpr int i = decltype(I)::value;
    static_for<TN>([&](auto J) {
      constexpr int j = decltype(J)::value;
      const floatx16 t = acc[i][j];
      static_for<4>([&](auto Q) {
        constexpr int qd = decltype(Q)::value;
        *reinterpret_cast<floatx4*>(region + (i * 32 + row32) * RBY + (((8 * j + 2 * qd + h) ^ (row32 & XM)) << 4)) =
            floatx4{t[4 * qd], t[4 * qd + 1], t[4 * qd + 2], t[4 * qd + 3]};
      });
    });
  });
  // Eight columns of a row per thread.
  constexpr int GROUPS = 128 * TM * TN, GPT = (GROUPS + NW * 64 - 1) / (NW * 64);
  const int waves = min(NW, KT);  // waves that had a K step
  typename AnyType<T>::template Epilogue<OutF32> epi(p, bz);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < GPT; ++u) {
    const int gidx = u * NW * 64 + tid;
    const int row = gidx / (4 * TN), c8 = gidx % (4 * TN);
    const int m = m0 + row, n = n0 + c8 * 8, count = p.N - n;
    if ((GROUPS % (NW * 64) == 0 || gidx < GROUPS) && m < p.M && count > 0) {
      epi.columns(n, count);
      const char* src = lds + row * RBY;
      const int lo = ((2 * c8) ^ (row & XM)) << 4, hi = ((2 * c8 + 1) ^ (row & XM)) << 4;
      floatx4 s0 = *reinterpret_cast<const floatx4*>(src + lo), s1 = *reinterpret_cast<const floatx4*>(src + hi);
      for (int w = 1; w < waves; ++w) {
        s0 += *reinterpret_cast<const floatx4*>(src + w * STAGE + lo);
        s1 += *reinterpret_cast<const floatx4*>(src + w * STAGE + hi);
      }
      float v[1][8] = {{s0[0], s0[1], s0[2], s0[3], s1[0], s1[1], s1[2], s1[3]}};
      epi.template apply<1>(v, {m}, n, count);
      store8<typename AnyType<T>::Out, OutF32>(member_out(p, bz), bz * p.sc + (int64_t)m * p.ldc + n, v[0], count);
    }
  }
}

// The kernel's variants, by index from kSlicesPolicy on in kPolicies.
template <typename T, bool OutF32, bool A_MC, bool B_MC, bool MIS>
void launch_slices_variant(int v, typename AnyType<T>::Params& p, int batch, hipStream_t st) {
  const Policy& pol = kPolicies[kSlicesPolicy + v];  // (fp8 has the same tiles under its own numbers)
  p.tiles_m = (int)xmk::ceil_div(p.M, pol.bm);
  p.tiles_n = (int)xmk::ceil_div(p.N, pol.bn);
  p.order = tile_order_slices((uint32_t)p.tiles_m, (uint32_t)p.tiles_n, p.K);
  const dim3 grid((unsigned)(p.tiles_m * p.tiles_n), 1, (unsigned)batch), block((unsigned)(pol.wgm * 64));
  switch (v) {
    case 0: hipLaunchKernelGGL((gemm_slices_kernel<T, OutF32, A_MC, B_MC, 1, 1, 4, MIS>), grid, block, 0, st, p); break;
    case 1: hipLaunchKernelGGL((gemm_slices_kernel<T, OutF32, A_MC, B_MC, 1, 1, 8, MIS>), grid, block, 0, st, p); break;
    case 2: hipLaunchKernelGGL((gemm_slices_kernel<T, OutF32, A_MC, B_MC, 1, 1, 16, MIS>), grid, block, 0, st, p); break;
    case 3: hipLaunchKernelGGL((gemm_slices_kernel<T, OutF32, A_MC, B_MC, 1, 2, 8, MIS>), grid, block, 0, st, p); break;
    case 4: hipLaunchKernelGGL((gemm_slices_kernel<T, OutF32, A_MC, B_MC, 2, 2, 4, MIS>), grid, block, 0, st, p); break;
    default: hipLaunchKernelGGL((gemm_slices_kernel<T, OutF32, A_MC, B_MC, 2, 2, 8, MIS>), grid, block, 0, st, p); break;
  }
}

template <typename T, bool OutF32, bool A_MC, bool B_MC>
void launch_slices_rows(int v, typename AnyType<T>::Params& p, int batch, hipStream_t st) {
  if (p.misaligned) launch_slices_variant<T, OutF32, A_MC, B_MC, true>(v, p, batch, st);
  else launch_slices_variant<T, OutF32, A_MC, B_MC, false>(v, p, batch, st);
}

template <typename T, bool OutF32>
void launch_slices_impl(bool a_mc, bool b_mc, int v, typename AnyType<T>::Params& p, int batch, hipStream_t st) {
  if (!a_mc && !b_mc) launch_slices_rows<T, OutF32, false, false>(v, p, batch, st);
  else if (!a_mc && b_mc) launch_slices_rows<T, OutF32, false, true>(v, p, batch, st);
  else if (a_mc && !b_mc) launch_slices_rows<T, OutF32, true, false>(v, p, batch, st);
  else launch_slices_rows<T, OutF32, true, true>(v, p, batch, st);
}

// Explicitly instantiated in gemm_inst_slices_*.hip.
template <typename T, bool OutF32>
void launch_slices(bool a_mc, bool b_mc, int v, typename AnyType<T>::Params& p, int batch, hipStream_t st);

}  // namespace gemm_impl
