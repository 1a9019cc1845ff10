// Int4 weight-only GEMM for more rows than one pass of int4_gemm_kernel takes (32): the same arithmetic -- exact
// integer weights on the matrix cores, scales and zero points applied per quantisation group to fp32 sums -- with
// the weights expanded in registers once per 32 or 64 rows.
//
//     out[m,n] = sum_g s[g,n] ( sum_{k in g} a[m,k] (16 + q[k,n])  -  (16 + z[g,n]) sum_{k in g} a[m,k] ) + bias[n]
//
// The offset that the expansion leaves on the weights is part of every sum up to the subtraction, so it has to be small:
// with 1024 + q, activations of one sign and zero points near the weights' mean the error against 64 bits was 2.37e-4
// (512 x 4096 x 16384), against 2.17e-4 of the kernel for few rows; with 16 + q it is 2.08e-4, which is the output's rounding
// (1.5 % of the results are not the nearest fp16 number; 30 % were).  No offset at all: nibbles as subnormal numbers lose
// bits inside the matrix instruction (10 % of the results), subtracting the offset in fp16 (0.1 %) took 91.6 us for 83.5.
//
// A work-group of NW waves owns 32 RT rows x 64 WN columns; WK = NW / WN waves take every WK-th 128 of K each and meet in
// LDS at the end, in wave order.  A wave owns 64 columns, two per lane: it loads two neighbouring packed words (eight k of
// two columns) at once and expands them into the operands of two 32x32x16 matrix instructions; no other wave of the
// work-group expands them again, and they are kept in registers for all row tiles.  The activations come in through LDS
// (two buffers, one step of 128 WK k each), the weights two steps ahead in registers.
//
// What bounds it: a wave's step of 128 k is 16 RT matrix instructions of 32 cycles, 128 vector instructions for the expansion
// (in the shadow of the former: up to six per matrix instruction cost nothing) and 32 RT for the scales.  The sums of a were
// 8 RT more matrix instructions of 32 cycles, whose 32 columns were all the same, and 32 RT more vector instructions took zero
// points off; now they are 16 RT of four by four, 8 cycles each and four in a row, since a change from one length to another costs
// ten cycles (one beside each product: 53 cycles a pair, no gain left), and one fp32 matrix instruction per two groups and 32 x 32
// results.  Their sums over the four waves that share rows, each a quarter of them, through LDS: no faster (82 us against 81).
// 512 x 4096 x 16384 at group 128 / 64 / 32: 91 -> 81 us, 104 -> 92, 163 -> 111; of the 81, 12 go with the power limit (69 on
// zeros) and 11 with staged activations, 8 are the launch, its first loads and its end.  Microseconds a call, weights from memory,
// group 128, against passes of 32 rows, each of which expands all weights, and against writing the fp16 weights out and the dense
// product on them: k 4096, n 16384: 64 rows 21.4 / 25.8 / 52.5, 128 29.6 / 50.6 / 55.9, 256 46.6 / 100 / 68.8, 512 81 / 199 / 93.3;
// k 16384, n 4096: 64 rows 33.2 / 41.6 / 76.4.
#include "int4_tile.h"

#include <type_traits>
#include <utility>

#include "common.h"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* lds_void_ptr;

constexpr uint32_t kOob = 0x80000000u;
constexpr int kStepK = 128;  // k a wave takes per step
constexpr int vmcnt_imm(int n) { return (n & 0xf) | ((n >> 4) << 14) | (0x7 << 4) | (0xf << 8); }

template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(static_cast<F&&>(f), std::make_integer_sequence<int, N>{});
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t r, char* lds, uint32_t voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_ptr)lds, 16, voff, 0, 0, 0);
}

// Two nibbles of a word, k = 2 i and 2 i + 1, as fp16 16 + q: times 2^6 + 2^18, a byte has its low nibble in bits 6 to 9 of
// the lower half and its high nibble in those of the upper one, where 0x4c00 | q << 6 is 16 + q.
__device__ __forceinline__ uint32_t expand(uint32_t w, int i, uint32_t magic) {
  return (__umul24((w >> (8 * i)) & 0xff, 0x00040040u) & 0x03c003c0u) | magic;
}
__device__ __forceinline__ float half_of(uint32_t pair, int c) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)(pair >> (16 * c)));
}

// Results of a finite row that are NaN, in columns with infinite scales: those come into the accumulators with a group's two
// sums one after the other, infinity less infinity, and are to come with their difference.  Formed again from the groups
// whose scale or zero point is not finite (the others do not matter beside them), in parts of 128 as the products are.
__device__ __forceinline__ void mend_columns(const xmk::Int4TileArgs& p, int m, int n, const half8& old, const float (&bias)[8]) {
  const _Float16* const a = p.act + (size_t)m * p.K;
  const int part = min(p.group, kStepK);
#pragma unroll 1
  for (int j = 0; j < 8; ++j) {
    if (old[j] == old[j]) continue;
    bool found = false;
    float sum = 0.f;
#pragma unroll 1
    for (int k0 = 0; k0 < p.K && sum == sum; k0 += part) {
      const size_t sz = (size_t)(k0 / p.group) * p.N + n + j;
      const float s = (float)p.scales[sz], z = (float)p.zeros[sz];
      if (fabsf(s) <= 65504.f && fabsf(z) <= 65504.f) continue;
      found = true;
      // (with an infinite zero point the weights do not matter)
      const bool far = !(fabsf(z) <= 65504.f);
      float diff = 0.f;
#pragma unroll 1
      for (int k = k0; k < k0 + part; ++k) {
        const float q = (float)((p.qw[(size_t)(k / 8) * p.N + n + j] >> (4 * (k % 8))) & 15);
        diff = fmaf((float)a[k], far ? 1.f : q - z, diff);
      }
      sum = fmaf(s, far ? -z * diff : diff, sum);
    }
    if (found) p.out[(size_t)m * p.N + n + j] = (_Float16)(sum + bias[j]);
  }
}

// An infinite activation makes both sums of its group infinite and their difference NaN, whatever the weights.  Eight results
// of a row that holds one, formed again weight by weight: the finite activations do not matter beside the others.
__device__ __forceinline__ void mend_row(const xmk::Int4TileArgs& p, int m, int n, const float (&bias)[8]) {
  _Float16* const out = p.out + (size_t)m * p.N + n;
  const half8 old = *reinterpret_cast<const half8*>(out);
  bool nan = false;
#pragma unroll
  for (int j = 0; j < 8; ++j) nan |= old[j] != old[j];
  if (!nan) return;
  bool found = false, open = true;  // open: not all eight are NaN yet
  float sum[8] = {};
#pragma unroll 1
  for (int r = 0; r < p.K / 8 && open; ++r) {
    const u32x4 a8 = *reinterpret_cast<const u32x4*>(p.act + (size_t)m * p.K + 8 * r);
#pragma unroll 1
    for (int i = 0; i < 8; ++i) {
      const uint32_t pair = i < 4 ? (i < 2 ? a8[0] : a8[1]) : (i < 6 ? a8[2] : a8[3]);
      const uint16_t bits = (uint16_t)(pair >> (16 * (i & 1)));
      if ((bits & 0x7c00) != 0x7c00) continue;
      found = true;
      const float a = (float)__builtin_bit_cast(_Float16, bits);
      const size_t sz = (size_t)(8 * r / p.group) * p.N + n;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float q = (float)((p.qw[(size_t)r * p.N + n + j] >> (4 * i)) & 15);
        sum[j] += a * ((q - (float)p.zeros[sz + j]) * (float)p.scales[sz + j]);
      }
      open = false;
#pragma unroll
      for (int j = 0; j < 8; ++j) open |= sum[j] == sum[j];
    }
  }
  if (!found) return mend_columns(p, m, n, old, bias);
  half8 o;
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = (_Float16)(sum[j] + bias[j]);
  *reinterpret_cast<half8*>(out) = o;
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
  constexpr bool kDefer = RT == 1;
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

  const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  floatx16 acc[RT][2];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) acc[rt][0] = acc[rt][1] = zero;
  uint32_t magic = 0x4c004c00u;
  asm volatile("" : "+v"(magic));  // (a value the compiler cannot see through: (x & m) | magic is then one instruction)
  const half4 ones = __builtin_bit_cast(half4, u32x2{0x3c003c00u, 0x3c003c00u});

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

  // A scale group's matrix instructions are a chain per row tile and column set; its sums go into acc with a multiply-add each.
  // What the offset and the zero point added to them comes off acc after every second group: an fp32 product of the row sums of two
  // groups, even and odd, with their s (16 + z).  acc holds it for two groups at most, so that next to nothing of its precision goes
  // to sums that cancel.  kDefer (32 rows): a chain's sums are worked in beside the next chain; 64 rows have no registers for that.
  floatx16 d[kDefer ? 2 : 1][RT][2];
  float sc[2][2], zz[2][2];  // of an even and an odd group: the scales, and -s (16 + z)
  float rows[2][RT];         // row sums over the lane's half of each k-step (a lane's column of a four by four product is its own,
                             // so that an infinite activation stays in its row)
  if constexpr (kDefer) {
    d[1][0][0] = d[1][0][1] = zero;
    sc[1][0] = sc[1][1] = 0.f;
  }
  auto fix_up = [&](auto P, auto E) {  // element E of the chains of parity P
    constexpr int par = decltype(P)::value, e = decltype(E)::value;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int c = 0; c < 2; ++c) acc[rt][c][e] = fmaf(sc[par][c], d[kDefer ? par : 0][rt][c][e], acc[rt][c][e]);
  };

  auto step = [&](auto ODD, int i, char* cur, char* next, Weights& w) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(kWeightLoads));  // this step's activations have landed; the next step's weights may be out
    __builtin_amdgcn_s_barrier();                         // for every wave, and the other buffer has been read
    __builtin_amdgcn_sched_barrier(0);
    half8 a[2][RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) a[0][rt] = fragment(cur, 0, rt);
    stage(i + 1, next);
    asm volatile("" : "+v"(magic) : : "memory");
    __builtin_amdgcn_sched_barrier(0);
    uint32_t b[2][2][4];
#pragma unroll
    for (int x = 0; x < 8; ++x) b[0][x / 4][x % 4] = expand(w.w[0][x / 4], x % 4, magic);
    static_for<NSUB>([&](auto U) {
      constexpr int u = decltype(U)::value, par = NSUB > 1 ? u & 1 : decltype(ODD)::value;
      floatx4 sum[2][RT];
      if constexpr (!kDefer) {
#pragma unroll
        for (int c = 0; c < 2; ++c) sc[par][c] = half_of(w.s[u], c);
      }
      static_for<SPG>([&](auto J) {
        constexpr int j = decltype(J)::value, s = u * SPG + j;
        static_for<2 * RT>([&](auto R) {
          constexpr int r = decltype(R)::value, rt = r / 2, c = r % 2;
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (s < 7 && c == 0) a[(s + 1) & 1][rt] = fragment(cur, s + 1, rt);
          auto& to = d[kDefer ? par : 0][rt][c];
          to = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[s & 1][rt], __builtin_bit_cast(half8, u32x4{b[s & 1][c][0], b[s & 1][c][1], b[s & 1][c][2], b[s & 1][c][3]}),
                                                      j == 0 ? zero : to, 0, 0, 0);
          if constexpr (s < 7) {
#pragma unroll
            for (int x = 4 * r / RT; x < 4 * (r + 1) / RT; ++x) b[(s + 1) & 1][x / 4][x % 4] = expand(w.w[s + 1][x / 4], x % 4, magic);
          }
          if constexpr (kDefer) {
            constexpr int slot = j * 2 * RT + r, slots = SPG * 2 * RT;
            static_for<16>([&](auto E) {
              constexpr int e = decltype(E)::value;
              if constexpr (e >= 16 * slot / slots && e < 16 * (slot + 1) / slots) fix_up(std::integral_constant<int, 1 - par>{}, E);
            });
          }
        });
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          const half8 v = a[s & 1][rt];
          const floatx4 none = {0.f, 0.f, 0.f, 0.f};
          sum[0][rt] = __builtin_amdgcn_mfma_f32_4x4x4f16(ones, __builtin_shufflevector(v, v, 0, 1, 2, 3), j == 0 ? none : sum[0][rt], 0, 0, 0);
          sum[1][rt] = __builtin_amdgcn_mfma_f32_4x4x4f16(ones, __builtin_shufflevector(v, v, 4, 5, 6, 7), j == 0 ? none : sum[1][rt], 0, 0, 0);
        }
      });
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        if constexpr (kDefer) sc[par][c] = half_of(w.s[u], c);
        zz[par][c] = fmaf(-sc[par][c], half_of(w.z[u], c), -16.f * sc[par][c]);
        asm volatile("" : "+v"(sc[par][c]), "+v"(zz[par][c]));  // (in registers of their own before the fetch below reuses w)
      }
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) rows[par][rt] = sum[0][rt][0] + sum[1][rt][0];
      if constexpr (u == NSUB - 1) fetch_pinned(i + 2, w);
      if constexpr (par == 1) {
        float off[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) off[c] = lane < 32 ? zz[0][c] : zz[1][c];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          // The upper lanes' half of the even group for the lower lanes' half of the odd one: the even group's sum then lies
          // in the lower lanes, the odd one's in the upper lanes.
          asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(rows[0][rt]), "+v"(rows[1][rt]));
          const float both = rows[0][rt] + rows[1][rt];
#pragma unroll
          for (int c = 0; c < 2; ++c) acc[rt][c] = __builtin_amdgcn_mfma_f32_32x32x2f32(both, off[c], acc[rt][c], 0, 0, 0);
        }
      }
      if constexpr (!kDefer) static_for<16>([&](auto E) { fix_up(std::integral_constant<int, par>{}, E); });
    });
  };

  Weights w0, w1;
  fetch(0, w0);
  stage(0, s0.stage);
  fetch_pinned(1, w1);
  typedef std::integral_constant<int, 0> Even;
  typedef std::integral_constant<int, 1> Odd;
  for (int i = 0; i < steps; i += 2) {  // (an odd count ends on a step of zeros)
    step(Even{}, i, s0.stage, s1, w0);
    step(Odd{}, i + 1, s1, s0.stage, w1);
  }
  if constexpr (kDefer) static_for<16>([&](auto E) { fix_up(Odd{}, E); });

  // Sums over the waves that split K, in wave order, one row tile after the other through LDS; a thread then owns eight
  // columns of a row.
  constexpr int TPR = BN / 8, RPP = NW * 64 / TPR;  // threads per row, rows per pass
  const int oc = (threadIdx.x % TPR) * 8, orow = threadIdx.x / TPR;
  float bias[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) bias[j] = p.bias && nb + oc < N ? (float)p.bias[nb + oc + j] : 0.f;
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // the loads past the end have landed too
  static_assert(32 % RPP == 0 || RT == 1, "a thread's rows are RPP apart over all row tiles");
  bool nan = false;  // one of this thread's results is
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
      for (int j = 0; j < 8; ++j) {
        o[j] = (_Float16)(v[j / 4][j % 4] + bias[j]);
        nan |= o[j] != o[j];
      }
      *reinterpret_cast<half8*>(p.out + (size_t)m * N + nb + oc) = o;
    }
  }
  if (__builtin_expect(nan, 0)) {
#pragma unroll 1
    for (int row = orow; row < BM; row += RPP)  // (the rows that this thread wrote)
      if (m0 + row < p.M && nb + oc < N) mend_row(p, m0 + row, nb + oc, bias);
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
  // Scales and zero points of groups of 32 are four times the work of those of 128 (512 x 4096 x 16384: 111 us where groups of
  // 128 take 81), the wide shapes' the most.
  const double g8 = group == 32 ? 1.15 : 1.0, g4 = group == 32 ? 1.25 : 1.0, gw = group == 32 ? 1.35 : group == 64 ? 1.1 : 1.0;
  Shape best = slim == 1 && k > 1024 ? Shape{Shape::kSlim8, 5.0 + 1.84 * g8 * steps(1024)}
                                     : Shape{Shape::kSlim4, 4.0 + 0.98 * g4 * steps(512) * (double)slim};
  const Shape others[] = {wide == 1 && k > 512 ? Shape{Shape::kWide8, 5.4 + 2.65 * gw * steps(512)}
                                               : Shape{Shape::kWide4, 4.6 + gw * steps(256) * pairs(wide, 2.5, 1.45)},
                          Shape{Shape::kBroad4, 4.6 + gw * steps(128) * pairs(broad, 2.35, 1.4)}};
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
