// FP8 (OCP e4m3fn) GEMM: out = bf16(d_scale * (a_scale * b_scale * A B + bias)), fp32 accumulation;
// d_scale and bias are optional.
//
// MFMA kernel: A [M,K] row-major and B stored [N,K] (both reduction-contiguous, the
// layout XLA's "__cublas$lt$matmul$f8" rewrite produces).  256x256 output tile per
// work-group (2x2 waves), K walked in steps of 64 bytes = one v_mfma_f32_32x32x64_f8f6f4
// k-step, in which a lane supplies 32 consecutive k of one row.  Operand tiles go from
// global memory straight into LDS (buffer_load ... lds) through the same 4-stage ring,
// swizzle and wait/barrier scheme as the 16-bit GEMM: a 64-byte fp8 row is byte for byte
// the 32-element 16-bit row that kernel's loader handles.  The per-tensor scales are read
// from device memory in the epilogue.
// B stored [K,N] (rhs_transpose == 0) takes the same kernel: its 64 k x BN tile goes into LDS as it
// lies in memory (n contiguous, the 16-bit GEMM's loader for that layout) and the fragments are read
// with ds_read_b64_tr_b8, which hands a lane 8 consecutive k of one column.
// Operands that the direct loads cannot take, and products with few output tiles, run the kernels that take any
// alignment (gemm_fp8.h).
#include <utility>

#include "gemm_fp8.h"

namespace gemm_impl {
// (gemm_inst_fp8_nk.hip / gemm_inst_fp8_kn.hip)
void launch_fp8_any_nk(int policy, Fp8Params& p, hipStream_t st);
void launch_fp8_any_kn(int policy, Fp8Params& p, hipStream_t st);
void launch_fp8_any(int policy, bool b_mc, Fp8Params& p, hipStream_t st) {
  if (b_mc) launch_fp8_any_kn(policy, p, st);
  else launch_fp8_any_nk(policy, p, st);
}
}  // namespace gemm_impl

namespace {

using gemm_impl::floatx16;
using gemm_impl::Fp8Epilogue;
using gemm_impl::Fp8Params;
using gemm_impl::intx8;
using gemm_impl::mfma_fp8;
using gemm_impl::static_for;
using gemm_impl::u32x2;
using gemm_impl::u32x4;
using gemm_impl::zero16;

constexpr uint32_t kOob = gemm_impl::kOob;

// Per-lane LDS byte offsets of an operand's fragments: lane l of the 32-row slab t gets row
// 32 t + l%32, bytes 64 ks + 32 (l/32) .. +31 of the row of BKB bytes, i.e. the two 16-byte chunks
// 4 ks + 2 (l/32) and + 1, each XOR-swizzled like the loader placed them.  Adding 32 t rows does not
// change the swizzle.
template <int BKB>
struct Fp8Frag {
  int base[BKB / 32];
  __device__ __forceinline__ void init(int row0, int lane) {
    const int row = row0 + (lane & 31);
    const int s = gemm_impl::swz<false, 0, BKB / 2>(row);
#pragma unroll
    for (int c = 0; c < BKB / 32; ++c) base[c] = row * BKB + (((c / 2 * 4 + (lane >> 5) * 2 + c % 2) ^ s) << 4);
  }
  __device__ __forceinline__ intx8 read(const char* __restrict__ tile, int t, int ks) const {
    const u32x4 lo = *reinterpret_cast<const u32x4*>(tile + base[2 * ks] + t * 32 * BKB);
    const u32x4 hi = *reinterpret_cast<const u32x4*>(tile + base[2 * ks + 1] + t * 32 * BKB);
    intx8 v;
    v[0] = (int)lo[0]; v[1] = (int)lo[1]; v[2] = (int)lo[2]; v[3] = (int)lo[3];
    v[4] = (int)hi[0]; v[5] = (int)hi[1]; v[6] = (int)hi[2]; v[7] = (int)hi[3];
    return v;
  }
};

// The same fragments from a tile stored [BKB k][BN columns] (row = BN bytes, 16-byte chunks XOR-swizzled
// by the loader with swz<true, BN / 2, 64, 1>(k)).  ds_read_b64_tr_b8 works on blocks of 16 lanes: lane p
// of a block addresses row kb + p / 2, bytes cb + 8 (p % 2) .. +7 and receives column cb + p, rows
// kb .. kb + 7.  Blocks 0 and 1 of the wave cover columns 0..15 and 16..31 of the slab for k half 0,
// blocks 2 and 3 the same columns for k half 1; four reads, 8 rows apart, give a lane its 32 k.  The
// swizzle depends on k & 7 = p / 2 only, so one address per slab serves the four reads.
template <int BN, int T>
struct Fp8FragKN {
  int base[T];
  __device__ __forceinline__ void init(int col0, int lane) {
    const int p = lane & 15;
    const int k = (lane >> 5) * 32 + (p >> 1);
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int col = col0 + t * 32 + ((lane >> 4) & 1) * 16 + 8 * (p & 1);
      base[t] = k * BN + (((col >> 4) ^ gemm_impl::swz<true, BN / 2, 64, 1>(k)) << 4) + (col & 15);
    }
  }
  // t counts 32-column slabs from col0; only slabs this wave owns are read.
  __device__ __forceinline__ intx8 read(const char* __restrict__ tile, int t, int ks) const {
    typedef int int2v __attribute__((ext_vector_type(2)));
    typedef int2v __attribute__((address_space(3))) * lds_ptr;
    intx8 v;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int2v r = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_ptr)(tile + base[t] + (ks * 64 + q * 8) * BN));
      v[2 * q] = r[0];
      v[2 * q + 1] = r[1];
    }
    return v;
  }
};

// BKB: bytes (k) of a K step, 64 or 128.
template <int BM, int BN, int WGM, int WGN, int NSTAGE, int BKB, bool BKN>
__global__ __launch_bounds__(WGM * WGN * 64) void fp8_gemm_kernel(Fp8Params p) {
  constexpr int NWAVES = WGM * WGN;
  constexpr int WTM = BM / WGM, WTN = BN / WGN;
  constexpr int TM = WTM / 32, TN = WTN / 32;
  constexpr int A_BYTES = BM * BKB, B_BYTES = BN * BKB, STAGE = A_BYTES + B_BYTES;
  constexpr int KS = BKB / 64;  // matrix instructions' k steps per K step
  // The loader works in 2-byte units.
  typedef gemm_impl::Loader<false, BM, BKB / 2, NWAVES> LoaderA;
  // B [n,k]: BN rows of BKB bytes; B [k,n]: BKB rows of BN bytes (BN / 2 two-byte units).
  typedef std::conditional_t<BKN, gemm_impl::Loader<true, BN / 2, BKB, NWAVES, 1>, gemm_impl::Loader<false, BN, BKB / 2, NWAVES>>
      LoaderB;
  constexpr int LOADS = LoaderA::NL + LoaderB::NL;  // per wave per K step
  static_assert(NSTAGE >= 3, "the barrier leaves the running step's loads in flight");
  __shared__ __attribute__((aligned(1024))) char lds[NSTAGE * STAGE];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;

  gemm_impl::request_first_args(p);
  const gemm_impl::TileAt tile = gemm_impl::tile_at(blockIdx.x, p.order);
  const int m0 = tile.m * BM, n0 = tile.n * BN;

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = zero16();

  LoaderA la;
  LoaderB lb;
  la.init(p.K / 2, p.M - m0, wave, lane);
  if constexpr (BKN) lb.init(p.N / 2, (p.N - n0) / 2, wave, lane);
  else lb.init(p.K / 2, p.N - n0, wave, lane);
  const uint8_t* a_tile = reinterpret_cast<const uint8_t*>(p.a) + (int64_t)m0 * p.K;
  const uint8_t* b_tile = reinterpret_cast<const uint8_t*>(p.b) + (BKN ? n0 : (int64_t)n0 * p.K);
  const int64_t b_step = BKN ? (int64_t)BKB * p.N : BKB;  // bytes from one K step's B tile to the next
  // k of a K step that exist, in the unit the loader compares with: two-byte units along a
  // k-contiguous row, rows of the [k,n] tile.
  auto kleft_b = [&](int st) { return BKN ? p.K - st * BKB : (p.K - st * BKB) / 2; };
  const int KT = (p.K + BKB - 1) / BKB;

  // Prologue: K steps 0 .. NSTAGE-2.  Loads past the end of K write zeros, so every step issues
  // the same number of loads and the vmcnt arithmetic is uniform.
#pragma unroll
  for (int st = 0; st < NSTAGE - 1; ++st) {
    la.issue(a_tile, (p.K - st * BKB) / 2, lds + st * STAGE, wave);
    lb.issue(b_tile, kleft_b(st), lds + st * STAGE + A_BYTES, wave);
    a_tile += BKB;
    b_tile += b_step;
  }
  __builtin_amdgcn_s_waitcnt(gemm_impl::vmcnt_imm((NSTAGE - 2) * LOADS));  // step 0 has landed
  __builtin_amdgcn_s_barrier();

  Fp8Frag<BKB> fa_addr;
  std::conditional_t<BKN, Fp8FragKN<BN, TN>, Fp8Frag<BKB>> fb_addr;
  fa_addr.init(wm * WTM, lane);
  fb_addr.init(wn * WTN, lane);
  // Fragment registers: the B fragments of a step are double-buffered (those of step kt + 1 are
  // read while step kt computes); the A fragments rotate through two slots, A fragment i + 1
  // being read under the MFMAs of fragment i, and fragment 0 of the next step under the last.
  static_assert(TM % 2 == 0 && TN <= TM, "fragment rotation");
  intx8 fa[2], fb[2][TN];
  constexpr int NMFMA = TM * TN;
  // One K step kt: B fragments (buffer `par`) and A fragment 0 of step kt are in registers.  Once
  // step kt + 1 has landed for every wave (vmcnt + barrier; all reads issued so far are complete
  // too), issue the loads of step kt + NSTAGE - 1 into the stage step kt - 1 used, and run the
  // MFMAs of step kt while reading the rest of its A fragments from `cur` and the first fragments
  // of step kt + 1 from `nxt`.  The stages are distinct (__restrict__), so the compiler keeps the
  // loads in flight across the fragment reads.
  auto k_step = [&](auto PAR, const char* __restrict__ cur, const char* __restrict__ nxt, char* __restrict__ wr,
                    int kt) {
    constexpr int par = decltype(PAR)::value;
    const int kleft = (p.K - (kt + NSTAGE - 1) * BKB) / 2;
    const __amdgpu_buffer_rsrc_t ra = gemm_impl::make_rsrc(a_tile), rb = gemm_impl::make_rsrc(b_tile);
    __builtin_amdgcn_s_waitcnt(gemm_impl::vmcnt_imm((NSTAGE - 3) * LOADS) & ~(0xf << 8));  // and lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int i = 0; i < LoaderA::NL; ++i) la.issue_one(i, ra, kleft, wr, wave);
#pragma unroll
    for (int i = 0; i < LoaderB::NL; ++i) lb.issue_one(i, rb, kleft_b(kt + NSTAGE - 1), wr + A_BYTES, wave);
    static_for<KS>([&](auto KSI) {
      constexpr int ks = decltype(KSI)::value, b = (par + ks) & 1;
      const char* const ahead = ks + 1 < KS ? cur : nxt;  // where the next k step's fragments are
      constexpr int nks = (ks + 1) % KS;
      static_for<TM>([&](auto I) {
        constexpr int i = decltype(I)::value;
        if constexpr (i + 1 < TM) fa[(i + 1) & 1] = fa_addr.read(cur, i + 1, ks);
        else fa[0] = fa_addr.read(ahead, 0, nks);
        if constexpr (i < TN) fb[b ^ 1][i] = fb_addr.read(ahead + A_BYTES, i, nks);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int jj = (i & 1) ? TN - 1 - j : j;  // boustrophedon: consecutive MFMAs share one operand
          acc[i][jj] = mfma_fp8(fb[b][jj], fa[i & 1], acc[i][jj]);
        }
      });
    });
    // Issue order: each row of MFMAs starts with its LDS reads (4 x 16 bytes), the global loads
    // are spread evenly.
    static_for<KS * NMFMA>([&](auto R) {
      constexpr int r = decltype(R)::value;
      if constexpr (r % TN == 0) __builtin_amdgcn_sched_group_barrier(0x100, (r / TN % TM < TN) ? (BKN ? 6 : 4) : 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if constexpr ((r + 1) * LOADS / (KS * NMFMA) > r * LOADS / (KS * NMFMA))
        __builtin_amdgcn_sched_group_barrier(0x020, (r + 1) * LOADS / (KS * NMFMA) - r * LOADS / (KS * NMFMA), 0);
    });
    __builtin_amdgcn_sched_barrier(0);
    a_tile += BKB;
    b_tile += b_step;
  };

#pragma unroll
  for (int j = 0; j < TN; ++j) fb[0][j] = fb_addr.read(lds + A_BYTES, j, 0);
  fa[0] = fa_addr.read(lds, 0, 0);
  for (int kt = 0; kt < KT; kt += 2) {
    k_step(std::integral_constant<int, 0>{}, lds + (kt % NSTAGE) * STAGE, lds + ((kt + 1) % NSTAGE) * STAGE,
           lds + ((kt + NSTAGE - 1) % NSTAGE) * STAGE, kt);
    if (kt + 1 < KT)
      k_step(std::integral_constant<int, KS & 1>{}, lds + ((kt + 1) % NSTAGE) * STAGE,
             lds + ((kt + 2) % NSTAGE) * STAGE, lds + ((kt + NSTAGE) % NSTAGE) * STAGE, kt + 1);
  }
  __builtin_amdgcn_s_waitcnt(gemm_impl::vmcnt_imm(0));  // drain the zero-fill loads before LDS is released

  // acc[i][j][e] is out[m][n], m = m0 + wm WTM + 32 i + lane%32, n = n0 + wn WTN + 32 j + 8 (e/4) + 4 (lane/32) + e%4.
  Fp8Epilogue epi(p);
  static_assert(NSTAGE * STAGE >= NWAVES * TN * 4096, "a slab per wave is staged in the operand stages");
  __builtin_amdgcn_s_barrier();  // every wave has read its last fragments
  gemm_impl::store_tile<__bf16, false>(epi, acc, lds + wave * (TN * 4096), p.out, p.N, 0, p.M, p.N, m0 + wm * WTM, n0 + wn * WTN, lane);
}

// Plain tiled kernel for operands of less than 16 bytes: 64x64 tile, fp8 decoded with the hardware
// conversion while staging, fp32 FMA.
__global__ __launch_bounds__(256) void fp8_gemm_generic_kernel(Fp8Params p, int rhs_transpose) {
  __shared__ float As[16][65];
  __shared__ float Bs[16][65];
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  float acc[4][4] = {};
  for (int k0 = 0; k0 < p.K; k0 += 16) {
    for (int e = threadIdx.x; e < 16 * 64; e += 256) {
      const int kk = e / 64, r = e % 64, k = k0 + kk;
      float av = 0.f, bv = 0.f;
      if (k < p.K && m0 + r < p.M)
        av = __builtin_amdgcn_cvt_f32_fp8((int)reinterpret_cast<const uint8_t*>(p.a)[(int64_t)(m0 + r) * p.K + k], 0);
      if (k < p.K && n0 + r < p.N) {
        const int64_t i = rhs_transpose ? (int64_t)(n0 + r) * p.K + k : (int64_t)k * p.N + (n0 + r);
        bv = __builtin_amdgcn_cvt_f32_fp8((int)reinterpret_cast<const uint8_t*>(p.b)[i], 0);
      }
      As[kk][r] = av;
      Bs[kk][r] = bv;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) { a[i] = As[kk][ty * 4 + i]; b[i] = Bs[kk][tx * 4 + i]; }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
  const Fp8Epilogue epi(p);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = m0 + ty * 4 + i, n = n0 + tx * 4 + j;
      if (m < p.M && n < p.N) reinterpret_cast<__bf16*>(p.out)[(int64_t)m * p.N + n] = epi(acc[i][j], n);
    }
}

// Up to 256 tiles of 128 x 128 a CU has one work-group, which may then fill its LDS: K steps of 128 bytes in four stages
// instead of 64.  Half the barriers, and whole cache lines from rows of k (268 instead of 366 MB at 256 x 16384 x 4096, B
// [n,k]).  Microseconds: there 22.8 -> 19.6, B [k,n] 23.5 -> 20.4; 512 x 4096 x 4096 19.3 -> 15.0, 128 x 16384 x 4096 20.2 ->
// 16.4.  (Three stages 25.2, five 20.9: neither the depth nor the barriers alone.)  With more tiles two work-groups share a CU,
// which the small stages allow: 700 x 6000 x 2048 18.3 against 19.9.  The 256 x 128 tile on steps of 128 bytes, three stages:
// 2048 x 4096 x 4096 37.9 -> 36.4 with B [n,k], 35.8 -> 36.8 with [k,n], 1024 x 8192 x 8192 74.9 -> 76.6: left alone.
bool one_per_cu(int64_t m, int64_t n) { return xmk::ceil_div(m, 128) * xmk::ceil_div(n, 128) <= 256; }

// XMK_FP8_POLICY=<index into kFp8Policies> forces a tile where the operands allow it (read at every call).
int choose_fp8(int64_t m, int64_t n, int64_t k, bool direct, bool any, bool rhs_t) {
  using namespace gemm_impl;
  auto usable = [&](int v) { return v >= 0 && v < kFp8Policies_n && (v < kFp8Direct ? direct : any); };
  if (const char* e = getenv("XMK_FP8_POLICY"))
    if (*e && usable(atoi(e))) return atoi(e);
  int best = -1;
  float best_cost = 1e30f;
  const uint32_t kt = (uint32_t)((k + 127) / 128);
  for (int pol = direct ? 0 : kFp8Direct; pol < kFp8Policies_n; ++pol) {
    if (!usable(pol)) continue;
    const TileCost& c = pol == 2 && one_per_cu(m, n) ? kFp8OnePerCu[rhs_t] : kFp8Cost[!direct ? 2 : rhs_t ? 1 : 0][pol];
    const float cost = launch_cost(kFp8Policies[pol], c, pol >= kFp8Slices, (uint32_t)m, (uint32_t)n, kt, 1);
    if (cost < best_cost) {
      best = pol;
      best_cost = cost;
    }
  }
  return best;
}

}  // namespace

extern "C" int xmk_fp8_gemm(const void* a, const void* b, const float* a_scale, const float* b_scale,
                            void* out, int64_t m, int64_t n, int64_t k, int32_t rhs_transpose,
                            void* stream) {
  return xmk_fp8_gemm_ex(a, b, a_scale, b_scale, nullptr, nullptr, out, m, n, k, rhs_transpose, stream);
}

extern "C" int xmk_fp8_gemm_ex(const void* a, const void* b, const float* a_scale, const float* b_scale,
                               const float* d_scale, const void* bias, void* out, int64_t m, int64_t n, int64_t k,
                               int32_t rhs_transpose, void* stream) {
  if (!a || !b || !a_scale || !b_scale || !out) return xmk::fail(XMK_INVALID_ARGUMENT, "fp8_gemm: null pointer");
  if (m <= 0 || n <= 0 || k <= 0) return xmk::fail(XMK_INVALID_ARGUMENT, "fp8_gemm: empty dimension");
  if (m > (1 << 30) || n > (1 << 30) || k > (1 << 30))
    return xmk::fail(XMK_INVALID_ARGUMENT, "fp8_gemm: dimension too large");
  Fp8Params p{};
  p.a = a; p.b = b; p.out = out; p.bias = bias;
  p.a_scale = a_scale; p.b_scale = b_scale; p.d_scale = d_scale;
  p.M = (int)m; p.N = (int)n; p.K = (int)k;
  p.lda = k; p.ldb = rhs_transpose ? k : n; p.ldc = n;
  p.alpha = 1.0f;
  hipStream_t st = (hipStream_t)stream;
  const bool aligned = xmk::aligned(a, 16) && xmk::aligned(b, 16) && k % 16 == 0 && p.ldb % 16 == 0;
  p.misaligned = !aligned;
  // The direct-to-LDS kernel: A rows and the stored rows of B start on 16-byte boundaries and hold whole
  // 16-byte chunks; one K step's tile of either operand lies within the 2 GiB a buffer descriptor spans.
  const bool direct = aligned && 256 * k < (int64_t)kOob && (rhs_transpose || 64 * n < (int64_t)kOob);
  // The tile loaders of the other kernels form byte offsets of up to 128 rows in 31 bits, from operands of 16 bytes
  // or more.
  const bool any = m * k >= 16 && n * k >= 16 && p.lda < (1 << 24) && p.ldb < (1 << 24);
  const int pol = choose_fp8(m, n, k, direct, any, rhs_transpose != 0);
  xmk::trace("fp8_gemm m=%lld n=%lld k=%lld rhs_t=%d -> %s", (long long)m, (long long)n, (long long)k, rhs_transpose,
             pol < 0 ? "generic_64x64" : gemm_impl::kFp8Policies[pol].name);
  if (pol >= gemm_impl::kFp8Direct) {
    gemm_impl::launch_fp8_any(pol, rhs_transpose == 0, p, st);
  } else if (pol >= 0) {
    const gemm_impl::Policy& P = gemm_impl::kFp8Policies[pol];
    p.tiles_m = (int)xmk::ceil_div(m, P.bm);
    p.tiles_n = (int)xmk::ceil_div(n, P.bn);
    p.order = gemm_impl::tile_order((uint32_t)p.tiles_m, (uint32_t)p.tiles_n, p.K);
    const dim3 grid((unsigned)(p.tiles_m * p.tiles_n)), block((unsigned)(P.wgm * P.wgn * 64));
    const bool kn = rhs_transpose == 0;
    if (pol == 0) {
      if (kn) hipLaunchKernelGGL((fp8_gemm_kernel<256, 256, 2, 4, 4, 64, true>), grid, block, 0, st, p);
      else hipLaunchKernelGGL((fp8_gemm_kernel<256, 256, 2, 4, 4, 64, false>), grid, block, 0, st, p);
    } else if (pol == 1) {
      if (kn) hipLaunchKernelGGL((fp8_gemm_kernel<256, 128, 2, 2, 4, 64, true>), grid, block, 0, st, p);
      else hipLaunchKernelGGL((fp8_gemm_kernel<256, 128, 2, 2, 4, 64, false>), grid, block, 0, st, p);
    } else if (one_per_cu(m, n)) {
      if (kn) hipLaunchKernelGGL((fp8_gemm_kernel<128, 128, 2, 2, 4, 128, true>), grid, block, 0, st, p);
      else hipLaunchKernelGGL((fp8_gemm_kernel<128, 128, 2, 2, 4, 128, false>), grid, block, 0, st, p);
    } else {
      if (kn) hipLaunchKernelGGL((fp8_gemm_kernel<128, 128, 2, 2, 4, 64, true>), grid, block, 0, st, p);
      else hipLaunchKernelGGL((fp8_gemm_kernel<128, 128, 2, 2, 4, 64, false>), grid, block, 0, st, p);
    }
  } else {
    hipLaunchKernelGGL(fp8_gemm_generic_kernel, dim3((unsigned)xmk::ceil_div(n, 64), (unsigned)xmk::ceil_div(m, 64)),
                       dim3(256), 0, st, p, (int)rhs_transpose);
  }
  return xmk::check_launch("fp8_gemm");
}
