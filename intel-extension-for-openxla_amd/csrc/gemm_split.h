// fp32 GEMM on the bf16 matrix instructions.  An fp32 number is the sum of three bf16 ones, exactly:
//     x = h + m + l,   h = bf16(x), m = bf16(x - h), l = x - h - m     (8 + 8 + 8 significant bits)
// and a product of two is h h' + (h m' + m h') + (h l' + m m' + l h') up to 2^-24 of itself, an fp32 rounding.  Six bf16 matrix
// instructions take the time of 3/8 of the fp32 ones: the device does 2.5 PFLOP/s in bf16 and 157 TFLOP/s in fp32.
//
// Error.  The bf16 instructions truncate what they align to the largest term, so that five small products added into the
// running sum of the large one bias it.  The large products of even and of odd halves of the K steps and the five small ones
// therefore have accumulators of their own, added at the end.
//
// Range.  Numbers are split times 2^23, which makes 2^-149, fp32's smallest, the smallest normal bf16: the parts of every number,
// however small, are normal or zero, and no product of them is lost.  (Numbers below 2^-102, which softmax weights and gradients have,
// were looked for before and their tiles formed again by the fp32 instructions: 2048 x 2048 x 1024 115 to 126 us.)  At the other end
// a number above 2^104 (h may be infinite) or an infinite one has a NaN for l, and so has a sum; a NaN shows the same way; a sum above
// 2^82 is not finite either.  The tile is then formed again by the fp32 instructions (gemm_ragged.h; all tiles of 2048 x 2048 x 1024
// 122 us).
//
// What bounds it: no unit alone.  24 products per wave and K step stand beside 110 vector instructions (6.5 per split number: each
// work-group splits what it loads), which share the issue port.  In a launch of one tile per CU the matrix pipe is busy 54 %
// of the time, vector and matrix instructions issue 44 %, LDS is busy 36 %, and the waves wait 29 % of theirs to issue and 31 % for
// data or the barrier.  Products and the rest are interleaved by hand in slots of one product, and a number's steps are spread
// over the slots, since what converts or subtracts has to wait for the one before.  The residuals by a shift or mask and a
// subtraction; v_dot2_f32_bf16, which does both at once, issues in ten cycles (1024 x 1024 x 4096 149 us, 122 without).
// Eight waves of 64 x 32; four of 64 x 64 read a third less from LDS and leave a SIMD with nothing beside a wait (165 us).
// 2048 x 2048 x 1024 71 -> 53 us (162 TFLOP/s where the fp32 instructions' peak is 157), 4096 x 4096 x 1024 252 -> 192,
// 3926 x 924 x 2976 192 -> 128.
//
// Error against 64 bits, of the result in the 2-norm, here / fp32 instructions on this tile:
//     k                        64               1024             4096             16384
//     normal                   4.4e-8 / 1.4e-7  1.3e-7 / 5.8e-7  2.7e-7 / 1.2e-6  5.8e-7 / 2.3e-6
//     uniform in 0 .. 1        4.0e-8 / 1.2e-7  8.6e-8 / 4.3e-7  1.6e-7 / 8.4e-7  3.0e-7 / 1.7e-6
//     normal, negatives 0      3.3e-8 / 6.5e-8  6.8e-8 / 2.5e-7  1.5e-7 / 4.9e-7  3.3e-7 / 9.9e-7
//     softmax x normal         6.5e-8 / 1.4e-7  1.5e-7 / 5.0e-7  2.8e-7 / 9.1e-7
// (on tiles whose waves split K the fp32 instructions reach 1.1e-7 / 1.6e-7 / 4.1e-7 for the first three of the first line).  Sums that
// one or two products make up are the other way round, as a truncated last place is twice a rounded one: e^(4 x), x normal, k 64
// and 256 6.9e-8 / 3.3e-8 and 1.1e-7 / 7.6e-8 (all elements alike, 8.9e-8 / 1.3e-7 and 1.0e-7 / 3.4e-7).
#pragma once
#include "gemm_ragged.h"

namespace gemm_impl {

constexpr float kSplitScale = 0x1p23f, kSplitUnscale = 0x1p-46f;

// AnyLoader's chunks of four floats, written to LDS as 3 planes of bf16: [row][32 k] (KC) or [k][rows] (MC), laid out and
// read as the 16-bit kernels' tiles with BK = 32.
template <bool MC, int ROWS, int NT, bool MIS>
struct SplitLoader : AnyLoader<float, MC, ROWS, NT, MIS> {
  typedef AnyLoader<float, MC, ROWS, NT, MIS> Base;
  typedef typename Base::Regs Regs;
  static constexpr int RB = MC ? ROWS * 2 : 64;  // bytes of an LDS row
  static constexpr int PLANE = ROWS * 64;
  static_assert(Base::RPL % (MC ? 4 : 16) == 0, "the swizzle repeats from load to load");
  int at;
  __device__ __forceinline__ void init(const float* op, int64_t ld, int row0, int rows, int64_t k0, int depth, int tid) {
    Base::init(op, ld, row0, rows, k0, depth, tid);
    const int row = tid / Base::CPR, c = tid % Base::CPR;
    at = row * RB + (((c >> 1) ^ swz<MC, ROWS, 32>(row)) << 4) + (c & 1) * 8;
    // (MC: chunks past the last column repeat the last one, as rows past the end do)
    if constexpr (MC) {
#pragma unroll
      for (int i = 0; i < Base::NL; ++i) this->off[i] -= 16 * max(c - (rows - 1 - row0) / 4, 0);
    }
  }
  // As the base's, with the lanes' offsets bounded in 32 bits (the compiler would do it in 64).
  __device__ __forceinline__ void load(Regs& r) {
    r.limit = (int32_t)min(this->left, (int64_t)0x7ffffff0);
    const char* from = r.limit < 0 ? this->base + r.limit : this->base;
    const uint32_t cap = (uint32_t)max(r.limit, 0);
#pragma unroll
    for (int i = 0; i < Base::NL; ++i) {
      uint32_t o;
      asm("v_min_u32 %0, %1, %2" : "=v"(o) : "s"(cap), "v"(this->off[i]));
      if constexpr (MIS) __builtin_memcpy(&r.g[i], from + o, 16);
      else r.g[i] = *reinterpret_cast<const u32x4*>(from + o);
    }
    this->advance(1);
  }
  // Zeroes what is no number of this tile: k from kleft on, (MC) columns from cleft on.  Chunks reach past both, into the padding
  // between a row's end and the next one or into the next row, and what lies there is neither looked at nor multiplied.
  __device__ __forceinline__ void clip(Regs& r, int kleft, int cleft) const {
    if (kleft >= Base::BK && (!MC || cleft >= ROWS)) return;  // (uniform)
    const int lrow = (int)threadIdx.x / Base::CPR, c = 4 * ((int)threadIdx.x % Base::CPR);
#pragma unroll
    for (int i = 0; i < Base::NL; ++i) {
      const int n = !MC ? kleft - c : lrow + i * Base::RPL < kleft ? cleft - c : 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) r.g[i][e] = e < n ? r.g[i][e] : 0u;
    }
  }
  // The numbers of a Regs on their way to LDS.  Pair q (elements 2 q and 2 q + 1) passes through seven steps, one after
  // the other; split_step<t>() runs step t - q of every pair that has it, so that a step's instructions do not wait for each other.
  static constexpr int PAIRS = 2 * Base::NL, STEPS = PAIRS + 6;
  struct Split {
    uint32_t part[3][PAIRS];
  };
  template <int STEP>
  __device__ __forceinline__ void split_step(char* tile, Regs& r, Split& s) const {
    typedef __bf16 v2 __attribute__((ext_vector_type(2)));
    static_for<PAIRS>([&](auto Q) {
      constexpr int q = decltype(Q)::value, step = STEP - q, i = q / 2, e = 2 * (q & 1);
      const float x0 = __builtin_bit_cast(float, (uint32_t)r.g[i][e]), x1 = __builtin_bit_cast(float, (uint32_t)r.g[i][e + 1]);
      if constexpr (step == 0) {
        r.g[i][e] = __builtin_bit_cast(uint32_t, x0 * kSplitScale);
        r.g[i][e + 1] = __builtin_bit_cast(uint32_t, x1 * kSplitScale);
      }
      if constexpr (step == 1 || step == 3 || step == 5) {
        s.part[step / 2][q] = __builtin_bit_cast(uint32_t, v2{(__bf16)x0, (__bf16)x1});
        asm("" : "+v"(s.part[step / 2][q]));  // (the compiler would convert x1 once more to have it alone)
      }
      if constexpr (step == 2 || step == 4) {  // what is left: exact
        const uint32_t h = s.part[step / 2 - 1][q];
        const float y0 = x0 - __builtin_bit_cast(float, h << 16);
        const float y1 = x1 - __builtin_bit_cast(float, h & 0xffff0000u);
        r.g[i][e] = __builtin_bit_cast(uint32_t, y0);
        r.g[i][e + 1] = __builtin_bit_cast(uint32_t, y1);
      }
      if constexpr (step == 6 && (q & 1)) {
#pragma unroll
        for (int pl = 0; pl < 3; ++pl)
          *reinterpret_cast<u32x2*>(tile + pl * PLANE + at + i * Base::RPL * RB) = u32x2{s.part[pl][q - 1], s.part[pl][q]};
      }
    });
  }
  __device__ __forceinline__ void store(char* tile, Regs& r, int kleft, int cleft) const {
    Split s;
    this->shift_ends(r);
    clip(r, kleft, cleft);
    static_for<STEPS>([&](auto S) { split_step<decltype(S)::value>(tile, r, s); });
  }
};

// BT x BT tile, 2 x WGN waves, K step of 32, two LDS stages of three planes per operand.
template <bool A_MC, bool B_MC, int BT, int WGN, bool MIS>
__global__ __launch_bounds__(2 * WGN * 64) void gemm_split_kernel(GemmParams p) {
  constexpr int BK = 32, KS = 2, NT = 2 * WGN * 64, TM = BT / 64, TN = BT / WGN / 32;
  typedef SplitLoader<A_MC, BT, NT, MIS> LoaderA;
  typedef SplitLoader<B_MC, BT, NT, MIS> LoaderB;
  constexpr int PLANE = LoaderA::PLANE, OP_BYTES = 3 * PLANE, STAGE = 2 * OP_BYTES;
  static_assert(2 * STAGE >= ragged_lds_bytes(BT) && 2 * STAGE >= 2 * WGN * TN * 4096, "also for the fp32 instructions and the epilogue");
  __shared__ __attribute__((aligned(1024))) char lds[2 * STAGE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;

  request_first_args(p);
  const TileAt tile = tile_at(blockIdx.x, p.order);
  const int m0 = tile.m * BT, n0 = tile.n * BT;
  const int64_t bz = blockIdx.z;
  const int64_t k0 = bz * p.kslice;  // K slices (kslice > 0): grid member z takes k0 .. k0 + kslice - 1
  const int K = p.kslice ? min(p.K - (int)k0, p.kslice) : p.K;
  LoaderA la;
  LoaderB lb;
  la.init(reinterpret_cast<const float*>(p.a) + bz * p.sa, p.lda, m0, p.M, k0, p.K, tid);
  lb.init(reinterpret_cast<const float*>(p.b) + bz * p.sb, p.ldb, n0, p.N, k0, p.K, tid);

  floatx16 acc[TM][TN], acc1[TM][TN], low[TM][TN];  // the products of the leading parts, by halves of the K steps; the other five
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = acc1[i][j] = low[i][j] = zero16();

  // Between the barriers of two K steps lie the second half of one step's matrix instructions and the first half of the
  // next one's: A of the step after that is split beside the former, B beside the latter, each into the stage that the
  // barrier has freed.  Loads are sent as soon as the registers are free, two K steps ahead; those past the end of K
  // come from the operand's last 16 bytes, and zeros are split in their place.
  const int cols_a = p.M - m0, cols_b = p.N - n0;
  typename LoaderA::Regs ga[2];  // K steps of even and odd number
  typename LoaderB::Regs gb[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    la.load(ga[i]);
    lb.load(gb[i]);
  }
  la.store(lds, ga[0], K, cols_a);
  la.load(ga[0]);
  lb.store(lds + OP_BYTES, gb[0], K, cols_b);
  lb.load(gb[0]);
  la.store(lds + STAGE, ga[1], K - BK, cols_a);
  la.load(ga[1]);
  lds_barrier();

  FragAddr<A_MC, BT, BK, TM> faddr;
  FragAddr<B_MC, BT, BK, TN> fbddr;
  faddr.init(wm * 32 * TM, lane);
  fbddr.init(wn * 32 * TN, lane);
  bf16x8 fa[2][3][TM], fb[2][3][TN];
  constexpr int READ_SLABS = 3 * (TM + TN);
  // Fragment f of a stage's half K step ks, in the order of their use.
  auto read_frag = [&](auto F, const char* stage, int ks) {
    constexpr int f = decltype(F)::value, pl = 2 - f / (TM + TN), i = f % (TM + TN);
    if constexpr (i < TM) fa[ks][pl][i] = faddr.template read<bf16x8>(stage + pl * PLANE, i, ks);
    else fb[ks][2 - pl][i - TM] = fbddr.template read<bf16x8>(stage + OP_BYTES + (2 - pl) * PLANE, i - TM, ks);
  };
  // Product r of a half K step's 6 TM TN, the smallest parts first.
  constexpr int NMFMA = 6 * TM * TN;
  constexpr int RSLOTS = (2 * NMFMA + 2) / 3, SSLOTS = (5 * NMFMA + 5) / 6;  // slots of a half K step with reads; with split numbers
  auto mma = [&](auto R, auto KSI) {
    constexpr int ks = decltype(KSI)::value, buf = ks, q = decltype(R)::value / (TM * TN), i = decltype(R)::value / TN % TM, j = decltype(R)::value % TN;
    constexpr int pa = q == 0 ? 2 : q == 1 || q == 3 ? 1 : 0, pb = q == 2 ? 2 : q == 1 || q == 4 ? 1 : 0;
    auto& to = q < 5 ? low : ks == 0 ? acc : acc1;
    to[i][j] = Elem<__bf16>::mfma(fb[buf][pb][j], fa[buf][pa][i], to[i][j]);
  };
  // Half a K step: its products, the reads of the next half's fragments (from the stage `frags`), and an operand's split numbers on
  // their way to LDS, in slots of one matrix instruction each.
  auto half = [&](auto KSI, auto CLIP, const char* frags, auto& ld, auto& regs, char* to, int kleft, int cleft) {
    constexpr int ks = decltype(KSI)::value;
    typedef std::remove_reference_t<decltype(ld)> L;
    typename L::Split s;
    ld.shift_ends(regs);
    if constexpr (decltype(CLIP)::value) ld.clip(regs, kleft, cleft);
    static_for<NMFMA>([&](auto R) {
      constexpr int r = decltype(R)::value;
      __builtin_amdgcn_sched_barrier(0);
      mma(R, KSI);
      constexpr int f0 = READ_SLABS * r / RSLOTS, f1 = READ_SLABS * (r + 1) / RSLOTS;
      static_for<READ_SLABS>([&](auto F) {
        constexpr int f = decltype(F)::value;
        if constexpr (f >= f0 && f < f1) read_frag(F, frags, 1 - ks);
      });
      constexpr int s0 = L::STEPS * r / SSLOTS, s1 = L::STEPS * (r + 1) / SSLOTS;
      static_for<L::STEPS>([&](auto S) {
        if constexpr (decltype(S)::value >= s0 && decltype(S)::value < s1) ld.template split_step<decltype(S)::value>(to, regs, s);
      });
      if constexpr (r == NMFMA - 1) ld.load(regs);
    });
    __builtin_amdgcn_sched_barrier(0);
  };
  const int KT = (K + BK - 1) / BK;
  static_for<READ_SLABS>([&](auto F) { read_frag(F, lds, 0); });
  typedef std::integral_constant<int, 0> First;
  typedef std::integral_constant<int, 1> Second;
  auto step = [&](auto ODD, auto CLIP, int kt) {
    constexpr int odd = decltype(ODD)::value, cur = odd * STAGE, nxt = STAGE - cur;
    half(First{}, CLIP, lds + cur, lb, gb[1 - odd], lds + nxt + OP_BYTES, K - (kt + 1) * BK, cols_b);
    lds_barrier();
    half(Second{}, CLIP, lds + nxt, la, ga[odd], lds + cur, K - (kt + 2) * BK, cols_a);
  };
  // Clipping costs 2 to 6 % of a step, so only the steps that split the last one's numbers do it (and all of a tile whose
  // last chunk of columns reaches past the end).
  const bool cut = (A_MC && cols_a < BT && cols_a % 4) || (B_MC && cols_b < BT && cols_b % 4);
  const int inside = cut ? 0 : (K - 2 * BK) / BK;  // whole K steps, two steps ago
  int kt = 0;
  for (; kt + 1 < inside; kt += 2) {
    step(First{}, std::false_type{}, kt);
    step(Second{}, std::false_type{}, kt + 1);
  }
  for (; kt + 1 < KT; kt += 2) {
    step(First{}, std::true_type{}, kt);
    if (kt + 2 < KT) step(Second{}, std::true_type{}, kt + 1);
  }
  const int cur = (KT - 1) % 2 * STAGE;
  static_for<READ_SLABS>([&](auto F) { read_frag(F, lds + cur, 1); });
  static_for<KS>([&](auto KSI) { static_for<NMFMA>([&](auto R) { mma(R, KSI); }); });
  bool redo = false;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      acc[i][j] += acc1[i][j] + low[i][j];
#pragma unroll
      for (int e = 0; e < 16; ++e) redo |= !(fabsf(acc[i][j][e]) <= 3.402823466e38f);
      acc[i][j] *= kSplitUnscale;
    }
  if (__syncthreads_or(redo)) ragged_products<float, A_MC, B_MC, BT, WGN, MIS>(p, m0, n0, bz, tid, lds, acc);

  lds_barrier();  // every wave has read its last fragments
  GemmEpilogue<float, true> epi(p, bz);
  store_tile<float, true>(epi, acc, lds + wave * (TN * 4096), member_out(p, bz), p.ldc, bz * p.sc, p.M, p.N, m0 + wm * 32 * TM,
                          n0 + wn * 32 * TN, lane);
}

// The tile of 64 stays with the fp32 instructions: four waves of 32 x 32 read LDS as often as they multiply, and a split
// one is 10 % slower at k = 128, level at 640 and where the large tile is faster than both by the time it gains.
template <bool A_MC, bool B_MC>
void launch_f32_tile(GemmParams& p, int batch, int tile, hipStream_t st) {
  p.tiles_m = (int)xmk::ceil_div(p.M, tile);
  p.tiles_n = (int)xmk::ceil_div(p.N, tile);
  p.order = tile_order((uint32_t)p.tiles_m, (uint32_t)p.tiles_n, p.K);
  const dim3 grid((unsigned)(p.tiles_m * p.tiles_n), 1, (unsigned)batch);
  auto go = [&](auto MIS) {
    constexpr bool mis = decltype(MIS)::value;
    if (tile == 128) hipLaunchKernelGGL((gemm_split_kernel<A_MC, B_MC, 128, 4, mis>), grid, dim3(512), 0, st, p);
    else hipLaunchKernelGGL((gemm_ragged_kernel<float, true, A_MC, B_MC, 64, 2, mis>), grid, dim3(256), 0, st, p);
  };
  p.misaligned ? go(std::true_type{}) : go(std::false_type{});
}

}  // namespace gemm_impl
