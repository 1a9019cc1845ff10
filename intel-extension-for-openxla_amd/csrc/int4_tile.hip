// Int4 weight-only GEMM for more rows than one pass of int4_gemm_kernel takes (32): the same arithmetic -- exact
// integer weights on the matrix cores, scales and zero points applied per quantisation group to fp32 sums -- with
// the weights expanded in registers once per 64 to 128 rows.
//
//     out[m,n] = sum_g s[g,n] ( sum_{k in g} a[m,k] (1024 + q[k,n])  -  (1024 + z[g,n]) sum_{k in g} a[m,k] ) + bias[n]
//
// A work-group of NW waves owns 32 RT rows x 64 WN columns; WK = NW / WN waves take every WK-th 128 of K each and meet in
// LDS at the end, in wave order.  A wave owns 64 columns, two per lane: it loads two neighbouring packed words (eight k of
// two columns) at once and expands them into the operands of two 32x32x16 matrix instructions; no other wave of the
// work-group expands them again, and they are kept in registers for all row tiles.  The activations come in through LDS
// (two buffers, one step of 128 WK k each), the weights two steps ahead in registers.
//
// What bounds it: a wave's step is 24 RT matrix instructions (16 RT of them the product, 8 RT the sums of a) and 176 vector
// instructions for the expansion, 64 RT for scales and zero points; with two waves per SIMD the matrix pipe is the longer of
// the two (512 x 4096 x 16384: 1.4 us per step), with one the two add up unless interleaved (kPipe: 64 rows in one row tile
// 24.4 -> 20.7 us with 32-row tiles).  Against passes of 32 rows, each of which expands all weights, and from 96 rows on
// against writing the fp16 weights out and the dense product on them (k 4096, n 16384): 64 rows 25.6 -> 20.7 us,
// 96 54.9 -> 26.9, 128 58.6 -> 28.3, 256 69.4 -> 47.1, 512 93.2 -> 87.8; k 16384, n 4096: 64 rows 40.6 -> 32.1,
// 128 84.7 -> 36.3.  Error against 64 bits 2.1e-4, the output's rounding (2.9e-4 where weights were rounded to fp16).
#include "int4_tile.h"

#include "common.h"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* lds_void_ptr;

constexpr uint32_t kOob = 0x80000000u;
constexpr int kStepK = 128;  // k a wave takes per step
constexpr int vmcnt_imm(int n) { return (n & 0xf) | ((n >> 4) << 14) | (0x7 << 4) | (0xf << 8); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t r, char* lds, uint32_t voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_ptr)lds, 16, voff, 0, 0, 0);
}

// The eight nibbles of a word as fp16 1024 + q, in the order of k.
__device__ __forceinline__ half8 expand(uint32_t w, uint32_t magic) {
  const uint32_t k04 = (w & 0x000f000fu) | magic, k15 = ((w >> 4) & 0x000f000fu) | magic;
  const uint32_t k26 = ((w >> 8) & 0x000f000fu) | magic, k37 = ((w >> 12) & 0x000f000fu) | magic;
  return __builtin_bit_cast(half8, u32x4{__builtin_amdgcn_perm(k15, k04, 0x05040100u), __builtin_amdgcn_perm(k37, k26, 0x05040100u),
                                         __builtin_amdgcn_perm(k15, k04, 0x07060302u), __builtin_amdgcn_perm(k37, k26, 0x07060302u)});
}
__device__ __forceinline__ float half_of(uint32_t pair, int c) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)(pair >> (16 * c)));
}

template <int STAGE, int NW>
union alignas(1024) StageOrSums {
  char stage[STAGE];
  float sums[NW * 32 * 64];  // one 32 x 64 tile per wave
};

// GS: k per scale and zero point inside a step (128 also for groups of 256: two steps read the same ones).
template <int RT, int WN, int NW, int GS>
__global__ __launch_bounds__(NW * 64, NW == 8 || (RT == 2 && WN > 1 && GS > 32) ? 2 : 1) void int4_tile_kernel(xmk::Int4TileArgs p) {
  constexpr int WK = NW / WN, BM = 32 * RT, BN = 64 * WN;
  constexpr int STAGE = BM * kStepK * 2 * WK;
  constexpr int RPL = 4 * NW, NI = BM / RPL;  // a staging load of all waves covers RPL rows: NI loads per wave and 128 of K
  constexpr int NSUB = kStepK / GS;        // scale groups per step
  constexpr int SPG = GS / 16;             // matrix instructions per scale group and tile
  constexpr bool kPipe = WN == 1 && NW == 4;
  constexpr int kWeightLoads = 8 + 2 * NSUB;
  static_assert(BM % RPL == 0, "whole loads");
  __shared__ StageOrSums<STAGE, NW> s0;
  __shared__ alignas(1024) char s1[STAGE];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave % WN, wk = wave / WN;
  // XCD x takes the x-th eighth of the tiles, the row blocks of a column block next to each other: they share its
  // weights in that XCD's L2.
  const int per_xcd = (int)gridDim.x / 8;
  const int item = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
  if (item >= p.row_blocks * p.col_blocks) return;
  const int m0 = item % p.row_blocks * BM, nb = item / p.row_blocks * BN;
  const int K = p.K, N = p.N;
  const int steps = (K + kStepK * WK - 1) / (kStepK * WK);

  // Every offset stands in the lane offset, which the hardware checks against the descriptor's size: rows, columns and k
  // past the end read as zeros.  (The host keeps all sums below 2^32.)
  const __amdgpu_buffer_rsrc_t r_a = make_rsrc(p.act + (size_t)m0 * K, (uint32_t)min(p.M - m0, BM) * (uint32_t)K * 2);
  const __amdgpu_buffer_rsrc_t r_w = make_rsrc(p.qw, (uint32_t)(K / 8) * (uint32_t)N * 4);
  const uint32_t sz_bytes = (uint32_t)(K / p.group) * (uint32_t)N * 2;
  const __amdgpu_buffer_rsrc_t r_s = make_rsrc(p.scales, sz_bytes), r_z = make_rsrc(p.zeros, sz_bytes);

  // staging: lane l of a wave takes chunk slot l % 16 of row RPL i + 4 wave + l / 16; chunk c of row r lies in slot
  // c ^ (r % 16), which spreads the 32 rows of a fragment read over all banks
  const int srow = 4 * wave + lane / 16, schunk = (lane % 16) ^ (srow % 16);
  const uint32_t voff_a = (uint32_t)(srow * K + schunk * 8) * 2;
  const int n0 = nb + 64 * wn + 2 * (lane % 32);
  const uint32_t voff_w = n0 < N ? (uint32_t)((lane / 32) * N + n0) * 4 : kOob;
  const uint32_t voff_s = n0 < N ? (uint32_t)n0 * 2 : kOob;

  auto stage = [&](int step, char* dst) {
#pragma unroll
    for (int j = 0; j < WK; ++j) {
      const int k0 = (step * WK + j) * kStepK;
      const bool in = k0 + schunk * 8 < K;
#pragma unroll
      for (int i = 0; i < NI; ++i)
        load_to_lds(r_a, dst + ((j * NI + i) * NW + wave) * 1024, in ? voff_a + (uint32_t)(RPL * i * K + k0) * 2 : kOob);
    }
  };
  struct Weights {
    u32x2 w[8];
    uint32_t s[NSUB], z[NSUB];
  };
  auto fetch = [&](int step, Weights& o) {
    const int k0 = min(step * WK + wk, (K - 1) / kStepK + 1) * kStepK;  // (past the end: the first step that lies there as a whole)
#pragma unroll
    for (int u = 0; u < NSUB; ++u) {
      const uint32_t so = (uint32_t)((k0 + u * GS) / p.group) * (uint32_t)N * 2;
      o.s[u] = __builtin_amdgcn_raw_buffer_load_b32(r_s, voff_s + so, 0, 0);
      o.z[u] = __builtin_amdgcn_raw_buffer_load_b32(r_z, voff_s + so, 0, 0);
    }
#pragma unroll
    for (int s = 0; s < 8; ++s)
      o.w[s] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r_w, voff_w + (uint32_t)(k0 / 8 + 2 * s) * (uint32_t)N * 4, 0, 0));
  };

  floatx16 acc[RT][2];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[rt][c][e] = 0.f;
  uint32_t magic = 0x64006400u;
  asm volatile("" : "+v"(magic));  // (a value the compiler cannot see through: (x & m) | magic is then one instruction)
  const half8 ones = __builtin_bit_cast(half8, u32x4{0x3c003c00u, 0x3c003c00u, 0x3c003c00u, 0x3c003c00u});

  // fragment of k-step s, row tile rt: row lane % 32, chunk 2 s + lane / 32
  const int frow = lane % 32;
  const uint32_t frag = (uint32_t)(wk * BM * 256 + frow * 256 + (((lane / 32) ^ (frow % 16)) << 4));

  auto fragment = [&](const char* cur, int s, int rt) {
    return *reinterpret_cast<const half8*>(cur + (frag ^ (uint32_t)(s << 5)) + rt * 8192);
  };
  // The waits on the staging loads count on this order: a step's staging loads, then the weights.
  auto fetch_pinned = [&](int step, Weights& w) {
    asm volatile("" : "+v"(magic) : : "memory");
    __builtin_amdgcn_sched_barrier(0);
    fetch(step, w);
    asm volatile("" : : : "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  // A chain of matrix instructions ends in 32 sums per lane that go into acc with two multiply-adds each.
  const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  struct Chain {
    floatx16 d[2], sum;
    float sc[2], zz[2];
  } last{{zero, zero}, zero, {0.f, 0.f}, {0.f, 0.f}};
  auto fix_up = [&](int rt, int from, int to) {
#pragma unroll
    for (int e = from; e < to; ++e)
#pragma unroll
      for (int c = 0; c < 2; ++c) acc[rt][c][e] = fmaf(last.sc[c], fmaf(last.zz[c], last.sum[e], last.d[c][e]), acc[rt][c][e]);
  };

  // kPipe (one wave per SIMD): the arithmetic between matrix instructions is spread over the chains -- the weights of a
  // k-step are expanded in front of its first use, a chain's sums are worked in during the next one -- since there is no
  // second wave to fill the gaps.
  auto step = [&](int i, char* cur, char* next, Weights& w) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(kWeightLoads));  // this step's activations have landed; the next step's weights may be out
    __builtin_amdgcn_s_barrier();                         // for every wave, and the other buffer has been read
    __builtin_amdgcn_sched_barrier(0);
    stage(i + 1, next);
    asm volatile("" : "+v"(magic) : : "memory");
    __builtin_amdgcn_sched_barrier(0);
    float sc[NSUB][2], zz[NSUB][2];
#pragma unroll
    for (int u = 0; u < NSUB; ++u)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        sc[u][c] = half_of(w.s[u], c);
        zz[u][c] = -1024.f - half_of(w.z[u], c);
        asm volatile("" : "+v"(sc[u][c]), "+v"(zz[u][c]));  // (in registers of their own before the fetch below reuses w)
      }
    half8 b[8][2];
    if constexpr (!kPipe) {
#pragma unroll
      for (int s = 0; s < 8; ++s)
#pragma unroll
        for (int c = 0; c < 2; ++c) b[s][c] = expand(w.w[s][c], magic);
      fetch_pinned(i + 2, w);
    }
    // chain q: scale group q / RT, row tile q % RT
    half8 a = fragment(cur, 0, 0);
#pragma unroll
    for (int q = 0; q < NSUB * RT; ++q) {
      const int u = q / RT, rt = q % RT, before = (q + RT - 1) % RT;
      floatx16 d0 = zero, d1 = zero, sum = zero;
#pragma unroll
      for (int j = 0; j < SPG; ++j) {
        const int s = u * SPG + j;
        if constexpr (kPipe) {
          if (rt == 0) {
            b[s][0] = expand(w.w[s][0], magic);
            b[s][1] = expand(w.w[s][1], magic);
          }
        }
        const int nj = (j + 1) % SPG, nq = nj == 0 ? q + 1 : q;
        const half8 now = a;
        if (nq < NSUB * RT) a = fragment(cur, nq / RT * SPG + nj, nq % RT);
        sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(now, ones, sum, 0, 0, 0);
        d0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(now, b[s][0], d0, 0, 0, 0);
        d1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(now, b[s][1], d1, 0, 0, 0);
        if constexpr (kPipe) {
          fix_up(before, j * 16 / SPG, (j + 1) * 16 / SPG);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      last.d[0] = d0; last.d[1] = d1; last.sum = sum;
#pragma unroll
      for (int c = 0; c < 2; ++c) last.sc[c] = sc[u][c], last.zz[c] = zz[u][c];
      if constexpr (!kPipe) fix_up(rt, 0, 16);
    }
    if constexpr (kPipe) fetch_pinned(i + 2, w);
  };

  Weights w0, w1;
  fetch(0, w0);
  stage(0, s0.stage);
  fetch_pinned(1, w1);
  for (int i = 0; i < steps; i += 2) {  // (an odd count ends on a step of zeros)
    step(i, s0.stage, s1, w0);
    step(i + 1, s1, s0.stage, w1);
  }
  if constexpr (kPipe) fix_up(RT - 1, 0, 16);

  // Sums over the waves that split K, in wave order, one row tile after the other through LDS; a thread then owns eight
  // columns of a row.
  constexpr int TPR = BN / 8, RPP = NW * 64 / TPR;  // threads per row, rows per pass
  const int oc = (threadIdx.x % TPR) * 8, orow = threadIdx.x / TPR;
  float bias[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) bias[j] = p.bias && nb + oc < N ? (float)p.bias[nb + oc + j] : 0.f;
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // the loads past the end have landed too
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int row = e % 4 + 8 * (e / 4) + 4 * (lane / 32);
      *reinterpret_cast<floatx2*>(&s0.sums[(wave * 32 + row) * 64 + 2 * (lane % 32)]) = floatx2{acc[rt][0][e], acc[rt][1][e]};
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < (31 + RPP) / RPP; ++r) {
      const int row = r * RPP + orow, m = m0 + rt * 32 + row;
      if (row >= 32 || m >= p.M || nb + oc >= N) continue;  // (N is a multiple of 8)
      floatx4 v[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int j = 0; j < WK; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          v[h] += *reinterpret_cast<const floatx4*>(&s0.sums[((j * WN + oc / 64) * 32 + row) * 64 + oc % 64 + 4 * h]);
      half8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (_Float16)(v[j / 4][j % 4] + bias[j]);
      *reinterpret_cast<half8*>(p.out + (size_t)m * N + nb + oc) = o;
    }
  }
}

template <int RT, int WN, int NW>
void launch_tile(xmk::Int4TileArgs p, hipStream_t st) {
  p.row_blocks = (int)xmk::ceil_div(p.M, 32 * RT);
  p.col_blocks = (int)xmk::ceil_div(p.N, 64 * WN);
  const dim3 grid((unsigned)(xmk::ceil_div((int64_t)p.row_blocks * p.col_blocks, 8) * 8)), block(NW * 64);
  if (p.group == 32) hipLaunchKernelGGL((int4_tile_kernel<RT, WN, NW, 32>), grid, block, 0, st, p);
  else if (p.group == 64) hipLaunchKernelGGL((int4_tile_kernel<RT, WN, NW, 64>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((int4_tile_kernel<RT, WN, NW, 128>), grid, block, 0, st, p);
}

// The tile shapes and what they cost.  All were timed at m 33 ... 1024 over k 1024 ... 16384 and n 1000 ... 16384; in
// microseconds a launch takes its base and, per step and round of work-groups (256, one per CU; two of the four-wave 64-row
// kinds share a CU and together take less than two rounds), the figures below.  A pair of steps is the unit of the K loop.
struct Shape {
  enum Kind { kSlim8, kSlim4, kWide8, kWide4, kBroad4 } kind;
  double us;
};
Shape choose(int64_t m, int64_t k, int64_t n, int64_t group) {
  auto steps = [&](int64_t per_step) { return (double)(xmk::ceil_div(k, 2 * per_step) * 2); };
  auto rounds = [&](int64_t rows, int64_t cols) { return xmk::ceil_div(xmk::ceil_div(m, rows) * xmk::ceil_div(n, cols), 256); };
  const int64_t slim = rounds(32, 64), wide = rounds(64, 128), broad = rounds(64, 256);
  auto pairs = [](int64_t r, double two, double one) { return (double)(r / 2) * two + (double)(r % 2) * one; };
  // 32 rows: few work-groups, so all eight waves on one reduction where there is a single round of them
  // (64 x 16384 x 4096: 32.1 us against 37.2; two rounds, 256 x 4096 x 4096: 22.7 against 19.2)
  // Scales and zero points of groups of 32 are four times the work of those of 128: 1.15 to 1.6 times the whole, the wide
  // shapes most (214 x 7264 x 5768: 83 us where groups of 128 take 51).
  const double g8 = group == 32 ? 1.15 : 1.0, g4 = group == 32 ? 1.35 : 1.0, gw = group == 32 ? 1.6 : 1.0;
  Shape best = slim == 1 && k > 1024 ? Shape{Shape::kSlim8, 5.0 + 1.95 * g8 * steps(1024)}
                                     : Shape{Shape::kSlim4, 4.0 + 1.03 * g4 * steps(512) * (double)slim};
  const Shape others[] = {wide == 1 && k > 512 ? Shape{Shape::kWide8, 5.4 + 2.85 * gw * steps(512)}
                                               : Shape{Shape::kWide4, 4.6 + gw * steps(256) * pairs(wide, 2.7, 1.65)},
                          Shape{Shape::kBroad4, 4.6 + gw * steps(128) * pairs(broad, 2.6, 1.7)}};
  for (const Shape& s : others)
    if (s.us < best.us) best = s;
  return best;
}

}  // namespace

bool xmk::int4_tile_applicable(const Int4TileArgs& p) {
  if (!p.act || !p.qw || !p.scales || !p.zeros || !p.out || p.M <= 0 || p.K <= 0 || p.N <= 0) return false;
  if (p.group != 32 && p.group != 64 && p.group != 128 && p.group != 256) return false;
  if (p.K % p.group != 0 || p.N % 8 != 0) return false;
  if (!aligned(p.act, 16) || !aligned(p.qw, 16) || !aligned(p.scales, 4) || !aligned(p.zeros, 4) || !aligned(p.out, 16)) return false;
  // 32-bit offsets: a block's rows, the weights and what a last step reaches past them (2^31 stands for "out of range" and
  // an offset is added to it), the number of tiles
  return p.M <= (1 << 16) && p.K <= (1 << 20) && p.N <= (1 << 20) && (uint64_t)(p.K / 8) * (uint64_t)p.N * 4 <= (1u << 30);
}

double xmk::int4_tile_cost(int64_t m, int64_t k, int64_t n, int64_t group) { return choose(m, k, n, group).us; }

void xmk::int4_tile_launch(const Int4TileArgs& p, hipStream_t st) {
  switch (choose(p.M, p.K, p.N, p.group).kind) {
    case Shape::kSlim8: launch_tile<1, 1, 8>(p, st); break;
    case Shape::kSlim4: launch_tile<1, 1, 4>(p, st); break;
    case Shape::kWide8: launch_tile<2, 2, 8>(p, st); break;
    case Shape::kWide4: launch_tile<2, 2, 4>(p, st); break;
    case Shape::kBroad4: launch_tile<2, 4, 4>(p, st); break;
  }
}
