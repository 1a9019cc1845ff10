// Fused multi-head attention forward for at most 128 keys: the cross attention of image models (77 text tokens) and
// short sequences.
//
// What bounds these calls is latency: the pipelined kernel (fmha_fwd_kernel.h) brings the queries in, then the keys
// half tile by half tile with a barrier per step, 10 us for [2,8,64,160] x 77 keys.  Here a work-group sends for its
// query rows and for ALL keys and values at once (one memory latency), forms every score of a row in registers,
// takes the row's exact maximum (no running reference, no rescale) and runs P V; two barriers in all.
// Layouts, fragments and the transposed products are those of fmha_fwd_kernel.h: a lane owns one query row.
// Pipelined kernel -> this one, back to back in a graph, f16: [2,8,64,160] x 77 keys 10.2 -> 6.6 us, [2,8,1024,80] x 77
// 7.1 -> 5.5, [4,20,4096,64] x 77 27.4 -> 22.4 (3.8 TB/s), [1,17,777,160] x 77 with a bias 21.0 -> 9.9.
// With a bias in 16-byte pieces ahead of the values (element by element and behind them before): 4 x 4 heads of 6446 x 40 and
// 77 keys 18.0 -> 12.4 us, 8 x 28 of 1118 x 40 31.1 -> 20.7, 2 x 26 of 614 x 160 18.4 -> 16.0.
#include "fmha_fwd_kernel.h"

namespace fmha_fwd_impl {
namespace {

// Chunk swizzles: 16 consecutive rows of one chunk column (K, Q) / 4 chunks of each of 4 consecutive rows (V) fall
// into different banks.
template <int CPR>
__device__ __forceinline__ int key_swizzle(int r) { return CPR % 16 == 0 ? (r & 15) : CPR == 8 ? ((r >> 1) & 7) : ((r >> 2) & 3); }
template <int CPR>
__device__ __forceinline__ int value_swizzle(int r) { return CPR % 16 == 0 ? (r & 3) << 2 : CPR == 8 ? (r & 2) << 1 : 0; }

// Load j of an operand tile: LDS bytes [1024 j, +1024); rows from `rows` on and h from H on read zeros.
template <int CPR, bool VALUES>
__device__ __forceinline__ void send(const void* base, int rows, int H, int j, char* tile) {
  const int idx = j * 64 + (threadIdx.x & 63), row = idx / CPR;
  const int chunk = (idx % CPR) ^ (VALUES ? value_swizzle<CPR>(row) : key_swizzle<CPR>(row));
  const uint32_t off = row < rows && chunk * 8 < H ? (uint32_t)((row * H + chunk * 8) * 2) : kOob;
  __builtin_amdgcn_raw_ptr_buffer_load_lds(make_rsrc(base, 0x7fffffffu), (lds_void_ptr)(tile + j * 1024), 16, off, 0, 0, 0);
}

// HP: head size padded to a multiple of 32; NKT: 32-key tiles; NW: waves, 32 query rows each.
template <typename T, int HP, int NKT, int NW, bool CAUSAL, bool BIAS>
__global__ __launch_bounds__(NW * 64) void fmha_short_kernel(FmhaParams p) {
  typedef typename Elem<T>::vec8 V8;
  constexpr int ROWB = HP * 2, CPR = HP / 8, KS = HP / 16, HT = HP / 32;
  constexpr int KV_BYTES = NKT * 32 * ROWB, Q_BYTES = 32 * ROWB;
  constexpr int NJ = KV_BYTES / 1024, NQ = Q_BYTES / 1024;  // 1 KiB loads of K (of V), and of a wave's queries
  __shared__ __attribute__((aligned(1024))) char lds[2 * KV_BYTES + NW * Q_BYTES];
  char* const k_tile = lds;
  char* const v_tile = lds + KV_BYTES;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, l32 = lane & 31;
  char* const q_tile = lds + 2 * KV_BYTES + wave * Q_BYTES;  // this wave's queries, later its output rows
  // The query blocks of a unit, which read the same keys, follow each other on one XCD.
  const int wg = (int)(blockIdx.x % 8) * p.per_xcd + (int)(blockIdx.x / 8);
  if (wg >= p.total) return;
  const int unit = wg / p.nqb, wq0 = (wg % p.nqb) * (NW * 32) + wave * 32;
  const int H = p.H, F = p.F, Tk = p.T;
  const int qrow = wq0 + l32;

  const T* Q = reinterpret_cast<const T*>(p.q) + ((int64_t)unit * F + wq0) * H;
  const T* K = reinterpret_cast<const T*>(p.k) + (int64_t)unit * Tk * H;
  const T* V = reinterpret_cast<const T*>(p.v) + (int64_t)unit * Tk * H;
#pragma unroll
  for (int j = 0; j < NQ; ++j) send<CPR, false>(Q, F - wq0, H, j, q_tile);
#pragma unroll
  for (int i = 0; i < (NJ + NW - 1) / NW; ++i)
    if (i * NW + wave < NJ) send<CPR, false>(K, Tk, H, i * NW + wave, k_tile);
  const bool active = wq0 < F;  // uniform over the wave
  // The bias of the wave's rows, sent for ahead of the values.
  u32x4 braw[BIAS ? NKT : 1][2];
  if constexpr (BIAS) {
    const int64_t first = (int64_t)unit * F;
    const int row = min(qrow, F - 1), last_row = min(wq0 + 31, F - 1);
    const T* bp = reinterpret_cast<const T*>(p.bias) + (first + row) * Tk + 16 * g;
    const int64_t after = ((int64_t)(p.total / p.nqb) * F - first - last_row) * Tk;  // elements behind key 0 of the last row
    if (active) {
#pragma unroll
      for (int t = 0; t < NKT; ++t) fetch_bias_keys(bp + 32 * t, 32 * t + 32 <= after, Tk - 32 * t - 16 * g, braw[t]);
    }
    asm volatile("" ::: "memory");
  }
#pragma unroll
  for (int i = 0; i < (NJ + NW - 1) / NW; ++i)
    if (i * NW + wave < NJ) send<CPR, true>(V, Tk, H, i * NW + wave, v_tile);

  floatx16 st[NKT];
#pragma unroll
  for (int t = 0; t < NKT; ++t) st[t] = zero16();
  // (Where a wave has one key tile the zeros are written here: behind the barrier they would be in the way, 8 x 25 heads of
  // 183 x 128 and 25 keys 6.83 us against 6.72.  With more tiles they hide behind each other's products: 8 x 28 of 6498 x 160
  // and 77 keys 266.8 us against 270.7 with the zeros here.)
  if constexpr (!BIAS && NKT == 1) asm volatile("" : "+v"(st[0]));

  // (the empty asm statements keep the compiler from moving LDS reads across)
  __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(NJ / NW));  // queries and keys have landed (a wave sent at least NJ / NW loads of V)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  V8 pf[NKT][2];
  float l_run = 0.0f, mref = 0.0f;
  if (active) {
    // Bias of the lane's 16 keys per tile: key 32 t + 8 (i / 4) + 4 g + i % 4.  (Keys past the end are masked below.)
    const float inv_scale = kLog2e / p.scale2;  // the bias is added in score units: (s + b / scale) * scale
    if constexpr (BIAS) {
#pragma unroll
      for (int t = 0; t < NKT; ++t) {
        u32x2 w[4];
        exchange_bias_keys(braw[t], w);
#pragma unroll
        for (int i = 0; i < 16; ++i) st[t][i] = bias_value<T>(w[i / 4], i % 4) * inv_scale;
      }
    }
    int kbase[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) kbase[s] = l32 * ROWB + (((2 * s + g) ^ key_swizzle<CPR>(l32)) << 4);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const V8 qf = __builtin_bit_cast(V8, *reinterpret_cast<const u32x4*>(q_tile + kbase[s]));
#pragma unroll
      for (int t = 0; t < NKT; ++t) {
        const u32x4 kf = *reinterpret_cast<const u32x4*>(k_tile + t * 32 * ROWB + kbase[s]);
        st[t] = Elem<T>::mfma(__builtin_bit_cast(V8, kf), qf, st[t]);
      }
    }
    // Mask (causal diagonal, end of the keys), row maximum.
    const int last = min(CAUSAL ? qrow : 0x7fffffff, Tk - 1) - 4 * g;  // largest visible key, less the lane's offset
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < NKT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        if (32 * t + 8 * (i / 4) + i % 4 > last) st[t][i] = -INFINITY;
        mx = __builtin_elementwise_maximum(mx, st[t][i]);
      }
    mx = __builtin_elementwise_maximum(mx, __shfl_xor(mx, 32));  // the lane with the row's other keys
    mref = mx == -INFINITY ? 0.0f : mx * p.scale2;
#pragma unroll
    for (int t = 0; t < NKT; ++t)
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const T r0 = (T)__builtin_amdgcn_exp2f(__builtin_fmaf(st[t][2 * k], p.scale2, -mref));
        const T r1 = (T)__builtin_amdgcn_exp2f(__builtin_fmaf(st[t][2 * k + 1], p.scale2, -mref));
        l_run = Elem<T>::dot2_ones(r0, r1, l_run);
        pf[t][k / 4][2 * (k % 4)] = r0;
        pf[t][k / 4][2 * (k % 4) + 1] = r1;
      }
  }
  __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if (!active) return;

  floatx16 ot[HT];
#pragma unroll
  for (int i = 0; i < HT; ++i) ot[i] = zero16();
  const int pl = lane & 15;
  auto accumulate = [&](auto TILES) {
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) {
      typedef short4v __attribute__((address_space(3))) * lds_ptr;
      const int col = 32 * ht + ((lane >> 4) & 1) * 16 + 4 * (pl & 3);
      const int key = 4 * g + (pl >> 2);  // + 8 for the second read, + 16 u + 32 t: none changes the swizzle
      const char* vb = v_tile + key * ROWB + (((col >> 3) ^ value_swizzle<CPR>(key)) << 4) + (col & 7) * 2;
#pragma unroll
      for (int t = 0; t < decltype(TILES)::value; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(vb + (32 * t + 16 * u) * ROWB));
          const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(vb + (32 * t + 16 * u + 8) * ROWB));
          u32x4 vv;
          vv[0] = __builtin_bit_cast(u32x2, lo)[0];
          vv[1] = __builtin_bit_cast(u32x2, lo)[1];
          vv[2] = __builtin_bit_cast(u32x2, hi)[0];
          vv[3] = __builtin_bit_cast(u32x2, hi)[1];
          ot[ht] = Elem<T>::mfma(__builtin_bit_cast(V8, vv), pf[t][u], ot[ht]);
        }
    }
  };
  // Causal: the tiles past the wave's rows are left out, not multiplied by weights of zero, since what lies there may be NaN.
  // One branch to straight-line code for each number of tiles (a branch around every tile: 2 to 9 % slower).
  if (CAUSAL && NKT > 1 && wq0 < 32) accumulate(std::integral_constant<int, 1>{});
  else if (CAUSAL && NKT > 2 && wq0 < 64) accumulate(std::integral_constant<int, (NKT > 2 ? 2 : 1)>{});
  else if (CAUSAL && NKT > 3 && wq0 < 96) accumulate(std::integral_constant<int, (NKT > 3 ? 3 : 1)>{});
  else accumulate(std::integral_constant<int, NKT>{});

  // O = O^T / l through the wave's own LDS rows, whole 16-byte chunks out; LSE = m + log l.
  const float l_tot = l_run + __shfl_xor(l_run, 32);
  const float inv = 1.0f / l_tot;
#pragma unroll
  for (int ht = 0; ht < HT; ++ht)
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
      union { T e[4]; u32x2 w; } r;
#pragma unroll
      for (int e = 0; e < 4; ++e) r.e[e] = (T)(ot[ht][4 * qd + e] * inv);
      *reinterpret_cast<u32x2*>(q_tile + l32 * ROWB + (((4 * ht + qd) ^ key_swizzle<CPR>(l32)) << 4) + g * 8) = r.w;
    }
  // (a row without a visible key: 0 + log 0; a row with a NaN: NaN)
  if (qrow < F && p.lse && g == 0) p.lse[(int64_t)unit * F + qrow] = mref * 0.6931471805599453f + logf(l_tot);
#pragma unroll 2
  for (int it = 0; it < NQ; ++it) {
    const int idx = it * 64 + lane, row = idx / CPR, c = idx % CPR;
    const u32x4 v = *reinterpret_cast<const u32x4*>(q_tile + row * ROWB + ((c ^ key_swizzle<CPR>(row)) << 4));
    if (wq0 + row < F && c * 8 < H)
      *reinterpret_cast<u32x4*>(reinterpret_cast<T*>(p.out) + ((int64_t)unit * F + wq0 + row) * H + c * 8) = v;
  }
}

template <typename T, int HP, bool CAUSAL, bool BIAS>
void launch_short_hp(FmhaParams p, uint64_t units, uint32_t F, hipStream_t st) {
  const int nkt = (p.T + 31) / 32;
  // (256 x 128 keys: K, V and four waves' queries would not fit the LDS)
  const int nw = HP == 256 && nkt == 4 ? 2 : 4;
  p.nqb = (int)((F + nw * 32 - 1) / (nw * 32));
  p.total = (int)(units * p.nqb);
  p.per_xcd = (p.total + 7) / 8;
  const dim3 grid((unsigned)(p.per_xcd * 8)), block(nw * 64);
  switch (nkt) {
    case 1: hipLaunchKernelGGL((fmha_short_kernel<T, HP, 1, 4, CAUSAL, BIAS>), grid, block, 0, st, p); break;
    case 2: hipLaunchKernelGGL((fmha_short_kernel<T, HP, 2, 4, CAUSAL, BIAS>), grid, block, 0, st, p); break;
    case 3: hipLaunchKernelGGL((fmha_short_kernel<T, HP, 3, 4, CAUSAL, BIAS>), grid, block, 0, st, p); break;
    default: hipLaunchKernelGGL((fmha_short_kernel<T, HP, 4, (HP == 256 ? 2 : 4), CAUSAL, BIAS>), grid, block, 0, st, p); break;
  }
}

template <typename T, bool CAUSAL, bool BIAS>
void launch_short_t(const FmhaParams& p, uint64_t units, uint32_t F, hipStream_t st) {
  if (p.H <= 64) launch_short_hp<T, 64, CAUSAL, BIAS>(p, units, F, st);
  else if (p.H <= 96) launch_short_hp<T, 96, CAUSAL, BIAS>(p, units, F, st);
  else if (p.H <= 128) launch_short_hp<T, 128, CAUSAL, BIAS>(p, units, F, st);
  else if (p.H <= 160) launch_short_hp<T, 160, CAUSAL, BIAS>(p, units, F, st);
  else launch_short_hp<T, 256, CAUSAL, BIAS>(p, units, F, st);
}

template <typename T>
void launch_short_t(const FmhaParams& p, uint64_t units, uint32_t F, bool causal, hipStream_t st) {
  // (Forms of their own with and without a bias: one form with a branch took 1 to 3 % longer without.)
  if (p.bias && causal) launch_short_t<T, true, true>(p, units, F, st);
  else if (p.bias) launch_short_t<T, false, true>(p, units, F, st);
  else if (causal) launch_short_t<T, true, false>(p, units, F, st);
  else launch_short_t<T, false, false>(p, units, F, st);
}

}  // namespace

void launch_short(const FmhaParams& p, int32_t dtype, uint64_t units, uint32_t F, bool causal, hipStream_t st) {
  if (dtype == XMK_BF16) launch_short_t<__bf16>(p, units, F, causal, st);
  else launch_short_t<_Float16>(p, units, F, causal, st);
}

}  // namespace fmha_fwd_impl
