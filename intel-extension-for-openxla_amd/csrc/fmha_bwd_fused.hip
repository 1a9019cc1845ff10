// Fused multi-head attention backward for bf16 / fp16 without a score-sized intermediate
// (the role of fmha_backward_kernel_{fp16,bf16}, xetla/sdp/sdp_backward.h:22-36).
//
// One kernel template, run with the roles of queries and keys exchanged:
//   owner = keys    : a work-group owns 128 keys (4 waves x 32) and walks the queries in blocks of 64;
//                     it accumulates dK = scale dS^T Q or dV = P^T dO for its keys (one launch each).
//   owner = queries : a work-group owns 128 queries and walks the keys; it accumulates dQ = scale dS K.
// with  P = exp(scale S - LSE),  dS = P o (dP - D),  S = Q K^T,  dP = dO V^T,  D = rowsum(dO o O).
// S (and dP) are recomputed in every pass (8 matrix products instead of 5) so that no gradient needs
// atomics or a second pass over partial sums: every output element is written once, in a fixed order.
// With scratch for it, and heads of more than 64, the owner = queries pass keeps dS, and dK takes it from there (6
// products; bwd_saved_pass).  Problems of few work-groups run all passes as one grid (one_grid() below).
//
// As in the forward kernel, every product is issued so that a lane owns ONE owner row:
//   scores  = Stream_tile . Owner^T : A operand = fragment of the streamed tile (LDS), B operand =
//             owner fragment (registers).  The 32x32 accumulator layout puts owner row l%32 in
//             lane l and the streamed rows in the lane's registers.
//   acc^T  += Stream_tile^T . dS    : the accumulator registers, converted, ARE the B operand (the
//             contraction runs over the streamed rows); the streamed tile is read with the LDS
//             transpose loads.
// The streamed tiles go from global memory straight into LDS, two stages.
#include <algorithm>
#include <utility>

#include "common.h"
#include "fmha_bwd_fused.h"

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* lds_void_ptr;

constexpr int BS = 64;   // streamed rows per block
constexpr int BO = 128;  // owner rows per work-group
constexpr uint32_t kOob = 0x80000000u;
// Cache policy of dS, written once and read once: 1079 -> 1034 us against the default ([8,32,2048,128] causal).
constexpr int kNonTemporal = 2;
constexpr float kLog2e = 1.4426950408889634f;

template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(static_cast<F&&>(f), std::make_integer_sequence<int, N>{});
}

template <typename T> struct Elem;
template <> struct Elem<__bf16> {
  typedef bf16x8 vec8;
  static __device__ __forceinline__ floatx16 mfma(vec8 a, vec8 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct Elem<_Float16> {
  typedef f16x8 vec8;
  static __device__ __forceinline__ floatx16 mfma(vec8 a, vec8 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

__device__ __forceinline__ floatx16 zero16() {
  return floatx16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ u32x4 buf_load(__amdgpu_buffer_rsrc_t r, uint32_t voff) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0));
}
// s_waitcnt immediate (gfx9 encoding): vmcnt(n), lgkmcnt(0), expcnt untouched.
__host__ __device__ constexpr int wait_vm_lgkm0(int n) { return (n & 0xf) | ((n >> 4) << 14) | (0x7 << 4); }

struct KParams {
  const void* own1;   // owner operand of the score product:   K (owner = keys) or Q
  const void* own2;   // owner operand of the dP product:      V (owner = keys) or dO
  const void* strm1;  // streamed operand of the score product: Q (owner = keys) or K
  const void* strm2;  // streamed operand of the dP product:    dO (owner = keys) or V
  const void* bias;   // [units, F, T] additive bias of the scores, or null
  int bias_vec;       // queries-own pass: the bias may be read 4 keys (8 bytes) at a time
  float* lse;         // [units, F] LSE of the forward pass times log2(e)    } the queries-own launch writes them and
  float* dsum;        // [units, F] D = rowsum(dO o O)                       } the keys-own ones read them; in one grid, all read
  const void* o;      // [units, F, H] forward output and
  const float* lse_fwd;  // [units, F] its LSE (queries-own launch)
  void* out1;         // scale * dS^T Q (dK)  or  scale * dS K (dQ)
  void* out2;         // P^T dO (dV), owner = keys only
  int H, F, T;
  int nob;            // owner blocks per unit
  int total, per_xcd, ug;
  float scale;
};
// (Apart: three sets of arguments go to the one grid of a small problem, which is 0.7 % faster without it over 400 drawn sizes.)
struct SavedParams : KParams {
  char* ds;  // dS of the launch's units (layout: ds_* below): the queries-own pass writes it, the saved-dS one reads it
};

// T: element type; HC: the head size that the products cover, 64, 96, 128, 160 or 256; HP: padded to 64, 128 or 256, the length
// of an LDS row (one wave per SIMD at 256); OWNER_K: the work-group owns keys (else queries).
// DS: accumulate out1 from dS (dK or dQ); PV: accumulate out2 from P (dV, owner = keys).  The
// keys-own work is run as two launches, one per output: with both accumulator sets and both owner
// operands a wave needs more than half the register file, and one wave per SIMD cannot overlap its
// matrix and vector work; recomputing S in a second launch at two waves per SIMD is faster.
// BIAS: S + bias enters the softmax; the bias is read from global memory at the start of each block
// (keys-own pass: 2-byte loads that are contiguous across the lanes of a wave; queries-own pass: each
// lane reads its own row, 8 bytes at a time where the alignment allows).
// STATS_IN: the row statistics are there (the queries-own pass reads them as the keys-own passes do, and writes none).
// SAVE_DS: the queries-own pass also writes dS, rounded as its own products take it, for bwd_saved_pass below.
// lds: bwd_lds_bytes(HP) bytes; block: the work-group's number among the pass's.

// Saved dS: tiles of 32 queries x 64 keys (4 KiB), a unit's tiles by blocks of 128 queries, in a block by 32 queries, then
// by keys; causal units hold no tiles past the diagonal block.  In a tile, the 16 bytes that a lane of the queries-own pass
// holds (query q, keys 16 u + 4 g + {0..3, 8..11}) are chunk (u / 2) 128 + (q / 4) 16 + (u % 2) 8 + 4 g + q % 4: a wave's
// store covers whole 128-byte lines, and the transpose reads of the saved-dS pass, which take 4 queries x 32 keys at a
// time, fall on 16 different chunks modulo the 256 bytes of the LDS banks.
constexpr int DS_TILE = 32 * BS * 2;
__host__ __device__ inline int ds_key_blocks(int T) { return (T + BO - 1) / BO * (BO / BS); }  // an even number
// Key blocks that the tiles of query block r cover, and how many tiles come before that block's.
__host__ __device__ inline int ds_width(int r, int nkb, bool causal) {
  const int w = (r + 1) * (BO / BS);
  return causal && w < nkb ? w : nkb;
}
__host__ __device__ inline int64_t ds_before(int r, int nkb, bool causal) {
  const int full = causal ? nkb / (BO / BS) : 0;  // blocks from here on are nkb wide
  const int64_t lo = r < full ? r : full;
  return (BO / 32) * (lo * (lo + 1) + (int64_t)(r - lo) * nkb);
}
// Bytes per unit.
inline size_t ds_unit_bytes(int F, int T, bool causal) {
  return (size_t)ds_before((F + BO - 1) / BO, ds_key_blocks(T), causal) * DS_TILE;
}

constexpr int padded(int HC) { return HC <= 64 ? 64 : HC <= 128 ? 128 : 256; }
constexpr int bwd_lds_bytes(int HP) { return 4 * BS * HP * 2 + 2 * (2 * BS * 4); }
template <typename T, int HC, bool OWNER_K, bool CAUSAL, bool DS, bool PV, bool BIAS, bool STATS_IN, bool SAVE_DS>
__device__ __forceinline__ void bwd_pass(const std::conditional_t<SAVE_DS, SavedParams, KParams>& p, char* lds, int block_id) {
  static_assert(DS || PV, "nothing to compute");
  static_assert(!SAVE_DS || !OWNER_K, "the queries-own pass saves dS");
  static_assert(!PV || OWNER_K, "P^T dO belongs to the keys-own pass");
  typedef typename Elem<T>::vec8 V8;
  constexpr int NW = 4;
  constexpr int HP = padded(HC);
  constexpr int ROWB = HP * 2;               // bytes of one tile row in LDS
  constexpr int CPR = ROWB / 16;             // 16-byte chunks per row
  constexpr int KMASK = 15;                  // the swizzle repeats every KMASK + 1 rows
  constexpr int TILE = BS * ROWB;
  constexpr int RPL = 1024 / ROWB;           // tile rows per 1 KiB load
  constexpr int NL = TILE / 1024 / NW;       // loads per wave per tile
  constexpr int LROWS = NW * RPL;            // tile rows between consecutive loads of a wave
  constexpr int KV = (LROWS % (KMASK + 1) == 0) ? 1 : 2;  // distinct swizzles among a wave's loads
  constexpr int KS = HC / 16;                // k-steps of the score products
  constexpr int HT = HC / 32;                // 32-wide h tiles of the gradients
  constexpr int STATS = 2 * BS * 4;          // LSE and D of one block's 64 query rows (owner = keys)
  static_assert(NL >= 1 && LROWS % 8 == 0 && (2 * LROWS) % (KMASK + 1) == 0, "tile / wave split");
  static_assert(bwd_lds_bytes(HP) == 4 * TILE + 2 * STATS, "what the kernels below reserve");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, l32 = lane & 31;
  // A tile row stores its 16-byte chunk c at position c ^ swz(row).  One tile serves two kinds of reads: row
  // fragments (16 lanes = 16 consecutive rows, one chunk column: swz must differ among 16 consecutive rows)
  // and transposed fragments (32 lanes = 4 consecutive rows x 4 adjacent chunks: bits 2-3 of swz must differ
  // among 4 consecutive rows, or the four rows land on the same banks).  Rows of 256 bytes and more: the two
  // bit pairs of row & 15, exchanged.  Rows of 128 bytes (8 chunks, two rows per 256 bytes of banks): the row's
  // parity already separates neighbours, and bits 1..3 of the row are dealt so that rows r and r + 2 differ in
  // bit 2 of swz and rows r and r + 8 in bit 1.
  auto swz = [](int row) {
    return CPR >= 16 ? (((row & 3) << 2) | ((row >> 2) & 3)) : ((((row >> 1) & 1) << 2) | ((row >> 2) & 3));
  };
  // Each XCD (own L2) gets a contiguous range of (unit, owner block) pairs: the owner blocks of a
  // unit stream the same tiles.
  const int wg = (block_id % 8) * p.per_xcd + block_id / 8;
  if (wg >= p.total || block_id >= 8 * p.per_xcd) return;
  // Inside the range, units go four at a time, owner blocks outermost and (causal) heaviest first, so that an
  // XCD's slots run dry at about the same time.
  const int UG = p.ug;
  const int ublk = wg / (UG * p.nob), r = wg % (UG * p.nob);
  const int gb = min(UG, p.total / p.nob - ublk * UG);  // units in this group (the last may hold fewer)
  const int unit = ublk * UG + r % gb;
  const int ob = OWNER_K ? r / gb : p.nob - 1 - r / gb;
  const int o0 = ob * BO;
  const int H = p.H;
  const int n_own = OWNER_K ? p.T : p.F;   // owner rows of the unit
  const int n_str = OWNER_K ? p.F : p.T;   // streamed rows of the unit

  const T* Own1 = reinterpret_cast<const T*>(p.own1) + (int64_t)unit * n_own * H;
  const T* Own2 = reinterpret_cast<const T*>(p.own2) + (int64_t)unit * n_own * H;
  const T* Str1 = reinterpret_cast<const T*>(p.strm1) + (int64_t)unit * n_str * H;
  const T* Str2 = reinterpret_cast<const T*>(p.strm2) + (int64_t)unit * n_str * H;
  float* lse = p.lse + (int64_t)unit * p.F;
  float* dsum = p.dsum + (int64_t)unit * p.F;

  // ---- owner fragments (B operands): this wave holds owner rows wo0 + l%32, fragment s covers
  // h = 16 s + 8 g .. +7.
  const int wo0 = o0 + wave * 32;
  const int orow = wo0 + l32;
  // They come in through LDS like the streamed tiles (below, once the tile loader is set up): read from global
  // memory in this layout, neighbouring lanes hold different rows, every lane is a cache access of its own, and
  // eight such loads per wave and operand cost the launch 18 us of load-path time at [8,32,2048,128].
  V8 of1[KS], of2[KS];
  // ---- streamed tile loads, global -> LDS, as in the forward kernel: load j = i * NW + wave fills
  // LDS bytes [1024 j, +1024) of the tile; lane l lands at row j * RPL + l / CPR, chunk l % CPR, and
  // fetches the global chunk that belongs there under the swizzle (swz below).
  const int lrow = wave * RPL + lane / CPR;
  uint32_t koff[KV];
#pragma unroll
  for (int v = 0; v < KV; ++v) {
    const int row = lrow + v * LROWS;
    const int chunk = (lane % CPR) ^ swz(row);
    koff[v] = chunk * 8 < H ? (uint32_t)((lrow * H + chunk * 8) * 2) : kOob;
  }
  const uint32_t lstride = (uint32_t)(LROWS * H * 2);
  auto issue_rows = [&](const T* base, int t0, char* __restrict__ tile, int n_rows) {
    const int rows_left = n_rows - t0;  // (<= 0: the whole tile is zeros)
    const __amdgpu_buffer_rsrc_t r = make_rsrc(base + (int64_t)t0 * H, 0x7fffffffu);
    const bool full = rows_left >= BS;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const uint32_t off = (full || lrow + i * LROWS < rows_left) ? koff[i % KV] : kOob;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_ptr)(tile + (i * NW + wave) * 1024), 16, off,
                                               i * lstride, 0, 0);
    }
  };
  auto issue_tile = [&](const T* base, int t0, char* __restrict__ tile) { issue_rows(base, t0, tile, n_str); };
  // LSE (waves 0, 2) and D (waves 1, 3) of the block's 64 query rows, one float per lane; rows past
  // F load zeros.  Every wave issues one load so that the load counts stay uniform.
  auto issue_stats = [&](int t0, char* __restrict__ st) {
    const float* src = (wave & 1) ? dsum : lse;
    const __amdgpu_buffer_rsrc_t r = make_rsrc(src, (uint32_t)p.F * 4);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_ptr)(st + (wave & 1) * (BS * 4)), 4,
                                             (uint32_t)((t0 + lane) * 4), 0, 0, 0);
  };

  // ---- per-lane LDS offsets of the fragments
  // Row fragment (kt, s): tile row 32 kt + l%32, logical chunk 2 s + g.
  int kbase[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) kbase[s] = l32 * ROWB + (((2 * s + g) ^ swz(l32)) << 4);
  // Transposed fragment (group u, h tile ht): two transpose reads; within a 16-lane block lane pl
  // addresses tile row 16 u + 4 g + pl/4 (+8 for the second read), h = cb + 4 (pl%4) .. +3.
  int tbase[HT][2];
  {
    const int pl = lane & 15;
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) {
      const int col = 32 * ht + ((lane >> 4) & 1) * 16 + 4 * (pl & 3);
      const int chunk = col >> 3, within = (col & 7) * 2;
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2) {
        const int row = 4 * g + (pl >> 2) + 8 * h2;  // + 16 u: does not change swz(row)
        tbase[ht][h2] = row * ROWB + ((chunk ^ swz(row)) << 4) + within;
      }
    }
  }

  floatx16 acc1[DS ? HT : 1], acc2[PV ? HT : 1];
#pragma unroll
  for (int i = 0; i < (DS ? HT : 1); ++i) acc1[i] = zero16();
#pragma unroll
  for (int i = 0; i < (PV ? HT : 1); ++i) acc2[i] = zero16();
  const float scale2 = p.scale * kLog2e;
  auto to_f32 = [](uint16_t b) -> float {
    if constexpr (sizeof(T) == 2 && __is_same(T, __bf16)) return __builtin_bit_cast(float, (uint32_t)b << 16);
    else return (float)__builtin_bit_cast(_Float16, b);
  };
  // Bias of one block in the layout of the scores: bs[kt][i] <-> streamed row t0 + 32 kt + 8 (i/4) + 4 g + i%4.
  auto load_bias = [&](int t0, float (&bs)[2][16]) {
    const T* bb = reinterpret_cast<const T*>(p.bias) + (int64_t)unit * p.F * p.T;
    const __amdgpu_buffer_rsrc_t r = make_rsrc(bb, (uint32_t)((int64_t)p.F * p.T * 2));
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const int s0 = t0 + 32 * kt + 8 * qd + 4 * g;  // first of 4 streamed rows
        if constexpr (OWNER_K) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int q = s0 + e;
            const uint32_t off = (q < p.F && orow < p.T) ? (uint32_t)(((int64_t)q * p.T + orow) * 2) : kOob;
            bs[kt][4 * qd + e] = to_f32((uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0));
          }
        } else {
          if (p.bias_vec) {  // T % 4 == 0: the 4 keys are inside the row or outside as a whole
            const uint32_t off = (orow < p.F && s0 < p.T) ? (uint32_t)(((int64_t)orow * p.T + s0) * 2) : kOob;
            const u32x2 w = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
#pragma unroll
            for (int e = 0; e < 4; ++e) bs[kt][4 * qd + e] = to_f32((uint16_t)(w[e >> 1] >> (16 * (e & 1))));
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const uint32_t off = (orow < p.F && s0 + e < p.T) ? (uint32_t)(((int64_t)orow * p.T + s0 + e) * 2) : kOob;
              bs[kt][4 * qd + e] = to_f32((uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0));
            }
          }
        }
      }
  };

  // Blocks of streamed rows this work-group needs.
  //   owner = queries, causal: keys up to its last query.   owner = keys, causal: queries from its first key on.
  const int b0 = (OWNER_K && CAUSAL) ? o0 / BS : 0;
  const int b1 = (!OWNER_K && CAUSAL) ? (min(n_str, o0 + BO) + BS - 1) / BS : (n_str + BS - 1) / BS;

  // D[streamed row][owner row] = Stream_tile . Owner^T for the 64 streamed rows of a block.
  auto scores = [&](const char* __restrict__ tile, const V8 (&of)[KS], floatx16 (&st)[2]) {
    st[0] = zero16();
    st[1] = zero16();
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        const u32x4 kv = *reinterpret_cast<const u32x4*>(tile + kbase[s] + kt * 32 * ROWB);
        st[kt] = Elem<T>::mfma(__builtin_bit_cast(V8, kv), of[s], st[kt]);
      }
  };
  // The same for the 32 streamed rows of half kt alone.
  auto scores_half = [&](const char* __restrict__ tile, const V8 (&of)[KS], int kt, floatx16& st) {
    st = zero16();
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const u32x4 kv = *reinterpret_cast<const u32x4*>(tile + kbase[s] + kt * 32 * ROWB);
      st = Elem<T>::mfma(__builtin_bit_cast(V8, kv), of[s], st);
    }
  };
  // acc^T += Stream_tile^T . F, with F given as four B-operand fragments (group u contracts the
  // streamed rows 16 u + {0..3, 8..11} + 4 g).
  auto accumulate = [&](const char* __restrict__ tile, const V8 (&fr)[4], floatx16 (&acc)[HT]) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int ht = 0; ht < HT; ++ht) {
        typedef short4v __attribute__((address_space(3))) * lds_ptr;
        const char* vt = tile + u * 16 * ROWB;
        const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(vt + tbase[ht][0]));
        const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(vt + tbase[ht][1]));
        u32x4 vv;
        vv[0] = __builtin_bit_cast(u32x2, lo)[0];
        vv[1] = __builtin_bit_cast(u32x2, lo)[1];
        vv[2] = __builtin_bit_cast(u32x2, hi)[0];
        vv[3] = __builtin_bit_cast(u32x2, hi)[1];
        acc[ht] = Elem<T>::mfma(__builtin_bit_cast(V8, vv), fr[u], acc[ht]);
      }
  };

  char* const s1 = lds;              // streamed tiles of the score product, two stages
  char* const s2 = lds + 2 * TILE;   // streamed tiles of the dP product, two stages
  char* const sst = lds + 4 * TILE;  // statistics, two stages

  // ---- owner fragments: the block's BO = 2 BS owner rows of each operand fill the two stages of s1 / s2; wave w
  // picks its 32 rows' fragments up as row fragments of tile w / 2, half w % 2.
  static_assert(BO == 2 * BS, "an owner block fills both stages");
  const char* const own_at = lds + (wave >> 1) * TILE + (wave & 1) * 32 * ROWB;
  issue_rows(Own1, o0, s1, n_own);
  issue_rows(Own1, o0 + BS, s1 + TILE, n_own);
  if constexpr (DS) {
    issue_rows(Own2, o0, s2, n_own);
    issue_rows(Own2, o0 + BS, s2 + TILE, n_own);
  }
  __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    of1[s] = __builtin_bit_cast(V8, *reinterpret_cast<const u32x4*>(own_at + kbase[s]));
    if constexpr (DS) of2[s] = __builtin_bit_cast(V8, *reinterpret_cast<const u32x4*>(own_at + 2 * TILE + kbase[s]));
  }
  __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));
  __builtin_amdgcn_s_barrier();  // every wave has its fragments: the stages may be overwritten
  // Softmax statistics of the lane's own query row (owner = queries): LSE log2(e) (one multiplication per row here
  // instead of one per score) and D = sum_h O[row][h] dO[row][h] (fmha_backward.h:48), formed from the dO fragments
  // the wave holds anyway and the same pieces of O, and written out for the keys-own launches that follow: a
  // separate pass over O and dO for them was 45 us at [8,32,2048,128].
  float own_lse2 = 0.f, own_d = 0.f;
  if constexpr (!OWNER_K && STATS_IN) {
    if (orow < p.F) {
      own_lse2 = lse[orow];
      own_d = dsum[orow];
    }
  } else if constexpr (!OWNER_K) {
    static_assert(DS, "the queries-own launch holds dO");
    const T* Oo = reinterpret_cast<const T*>(p.o) + (int64_t)unit * n_own * H;
    issue_rows(Oo, o0, s1, n_own);
    issue_rows(Oo, o0 + BS, s1 + TILE, n_own);
    __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));
    __builtin_amdgcn_s_barrier();
    float part = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const u32x4 ow = *reinterpret_cast<const u32x4*>(own_at + kbase[s]);
      const T* oe = reinterpret_cast<const T*>(&ow);
      const T* de = reinterpret_cast<const T*>(&of2[s]);
#pragma unroll
      for (int e = 0; e < 8; ++e) part += (float)oe[e] * (float)de[e];
    }
    own_d = part + __shfl_xor(part, 32);  // the row's other eight-element pieces are in lane l ^ 32
    if (orow < p.F) {
      own_lse2 = p.lse_fwd[(int64_t)unit * p.F + orow] * 1.4426950408889634f;
      if (g == 0) {
        lse[orow] = own_lse2;
        dsum[orow] = own_d;
      }
    }
    __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));
    __builtin_amdgcn_s_barrier();
  }


  // This wave's tiles of dS, and the lane's chunk in each.
  [[maybe_unused]] __amdgpu_buffer_rsrc_t ds_rsrc;
  [[maybe_unused]] const uint32_t ds_lane = (l32 >> 2) * 256 + g * 64 + (l32 & 3) * 16;
  if constexpr (SAVE_DS) {
    const int nkb = ds_key_blocks(p.T), w = ds_width(ob, nkb, CAUSAL);
    ds_rsrc = make_rsrc(p.ds + (int64_t)DS_TILE * (unit * ds_before(p.nob, nkb, CAUSAL) + ds_before(ob, nkb, CAUSAL) + (int64_t)wave * w),
                        (uint32_t)w * DS_TILE);
  }

  // One block: its tiles are in `c1`, `c2`, `cst`; the next block's go to `n1`, `n2`, `nst`.
  auto block = [&](int it, const char* __restrict__ c1, const char* __restrict__ c2, const char* __restrict__ cst,
                   char* __restrict__ n1, char* __restrict__ n2, char* __restrict__ nst) {
    const int t0 = it * BS;
    if (it + 1 < b1) {
      issue_tile(Str1, t0 + BS, n1);
      issue_tile(Str2, t0 + BS, n2);
      if constexpr (OWNER_K) issue_stats(t0 + BS, nst);
    }
    float bs[BIAS ? 2 : 1][16];
    if constexpr (BIAS) load_bias(t0, bs);
    // With both owner operands and the accumulators of the larger head sizes there are registers for the scores of half a
    // block: one half's are dead before the other's are made.  (A whole block's: the dK launch spills 30 registers, the
    // dQ launch has none left in which to read fragments ahead of their products, 526 -> 499 us at [8,32,2048,128] causal; with a
    // bias, whose loads the second half then waits for, it is faster whole: 40 heads of 459 x 128 94.6 us, by halves 101.3.)
    constexpr bool BY_HALF = DS && HP >= 128 && (OWNER_K || !BIAS || HP > 128);
    floatx16 sc[2], dp[2];
    if constexpr (!BY_HALF) {
      scores(c1, of1, sc);
      if constexpr (DS) scores(c2, of2, dp);
    }
    // sc[kt][i], dp[kt][i] <-> streamed row t0 + 32 kt + 8 (i/4) + 4 g + i%4, owner row `orow`.
    V8 pf[4], df[4];
    // Blocks that end inside the streamed range and (causal) lie wholly on the visible side of the
    // diagonal for every row of this wave need no mask (wave-uniform test).
    const bool masked = t0 + BS > n_str || (CAUSAL && (OWNER_K ? wo0 + 31 > t0 : t0 + BS - 1 > wo0));
    auto elementwise = [&](auto MASKED_T, auto KT_LO, auto KT_HI) {
      constexpr bool MASKED = decltype(MASKED_T)::value;
#pragma unroll
      for (int kt = decltype(KT_LO)::value; kt < decltype(KT_HI)::value; ++kt)
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
          floatx4 l2, dd;
          if constexpr (OWNER_K) {
            l2 = *reinterpret_cast<const floatx4*>(cst + (32 * kt + 8 * qd + 4 * g) * 4);
            dd = *reinterpret_cast<const floatx4*>(cst + BS * 4 + (32 * kt + 8 * qd + 4 * g) * 4);
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int i = 4 * qd + e;
            const float lse2 = OWNER_K ? l2[e] : own_lse2;
            const float dq = OWNER_K ? dd[e] : own_d;
            float arg;
            if constexpr (BIAS) arg = __builtin_fmaf(sc[kt][i], scale2, __builtin_fmaf(bs[kt][i], kLog2e, -lse2));
            else arg = __builtin_fmaf(sc[kt][i], scale2, -lse2);
            if constexpr (MASKED) {
              // The mask goes into the exponent (a select on a ready value, exp2(-inf) = 0): with `pr = 0` after
              // the exponential the compiler branches around every single exponential instead.
              const int srow = t0 + 32 * kt + 8 * qd + 4 * g + e;
              const int q = OWNER_K ? srow : orow;
              const int key = OWNER_K ? orow : srow;
              arg = (srow >= n_str || (CAUSAL && key > q)) ? -INFINITY : arg;
            }
            const float pr = __builtin_amdgcn_exp2f(arg);
            // fragment u = 2 kt + (qd >> 1) holds registers 8 (u & 1) .. +7 of tile kt
            if constexpr (PV) pf[2 * kt + (qd >> 1)][4 * (qd & 1) + e] = (T)pr;
            if constexpr (DS) df[2 * kt + (qd >> 1)][4 * (qd & 1) + e] = (T)(pr * (dp[kt][i] - dq));
          }
        }
    };
    typedef std::integral_constant<int, 0> i0;
    typedef std::integral_constant<int, 1> i1;
    typedef std::integral_constant<int, 2> i2;
    if constexpr (BY_HALF) {
      scores_half(c1, of1, 0, sc[0]);
      scores_half(c2, of2, 0, dp[0]);
      if (masked) elementwise(std::true_type{}, i0{}, i1{});
      else elementwise(std::false_type{}, i0{}, i1{});
      scores_half(c1, of1, 1, sc[1]);
      scores_half(c2, of2, 1, dp[1]);
      if (masked) elementwise(std::true_type{}, i1{}, i2{});
      else elementwise(std::false_type{}, i1{}, i2{});
    } else {
      if (masked) elementwise(std::true_type{}, i0{}, i2{});
      else elementwise(std::false_type{}, i0{}, i2{});
    }
    if constexpr (SAVE_DS) {
      // Rows past the last query hold what zeros make of the keys, which is NaN where a key holds an infinity or a NaN; the pass
      // that reads dS adds it, times zero, to that key's gradient.
      if (wo0 + 31 >= p.F) {
#pragma unroll
        for (int u = 0; u < 4; ++u) df[u] = orow < p.F ? df[u] : V8{};
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, df[u]), ds_rsrc, ds_lane,
                                               it * DS_TILE + (u >> 1) * 2048 + (u & 1) * 128, kNonTemporal);
    }
    if constexpr (DS) accumulate(c1, df, acc1);
    if constexpr (PV) accumulate(c2, pf, acc2);
    // The next block's tiles have landed (this wave's loads; every wave's after the barrier), and
    // this wave is done reading the tiles that the loads after the next block overwrite.  The stores of dS, issued
    // after those loads, are left in flight.
    __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(SAVE_DS ? 4 : 0));
    __builtin_amdgcn_s_barrier();
  };

  if (b0 < b1) {
    issue_tile(Str1, b0 * BS, s1);
    issue_tile(Str2, b0 * BS, s2);
    if constexpr (OWNER_K) issue_stats(b0 * BS, sst);
    __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));
    __builtin_amdgcn_s_barrier();
    // Two blocks a turn: with the stages picked by a block's parity instead, the two copies of the block met at every turn, and
    // the accumulators were moved from one's registers to the other's (64 moves a block; 4 heads of 4096 x 128 154 -> 129 us
    // together with the half blocks, 16 x 2048 heads of 64 157 -> 146, 32 x 4096 of 160 913 -> 821).
    // Heads above 128: up to four blocks go one a turn, since leaving such a turn in its middle moves accumulators, which a
    // short pass has nothing to set against (30 heads of 187 x 256 causal 27.2 -> 24.9 us).  With the short loop in front the compiler
    // also finds better registers for the long one: 32 x 1024 heads of 256 causal 163.6 -> 138.5, of 160 105.8 -> 96.8.
    // So do all passes of heads up to 128 with a bias (128 heads of 1024 x 64 218 us, with two blocks a turn 242; 40 of 459 x 80 85.2
    // and 89.6; over 70 drawn sizes of heads of 80 to 128 level on the mean, from 10 % slower to 8 % faster), and those of heads above
    // 160 with a bias and no mask (38 heads of 148 x 192 77.9 us, with both loops 81.4; 34 sizes 2 % on the mean; causal ones
    // and heads of 160 are 5 to 8 % faster with both).
    if ((HP > 128 && b1 - b0 <= 4) || (BIAS && (HP <= 128 || (HP > 160 && !CAUSAL)))) {
      for (int it = b0; it < b1; ++it) {
        if ((it - b0) & 1) block(it, s1 + TILE, s2 + TILE, sst + STATS, s1, s2, sst);
        else block(it, s1, s2, sst, s1 + TILE, s2 + TILE, sst + STATS);
      }
    } else
    for (int it = b0; it < b1; it += 2) {
      block(it, s1, s2, sst, s1 + TILE, s2 + TILE, sst + STATS);
      if (it + 1 < b1) block(it + 1, s1 + TILE, s2 + TILE, sst + STATS, s1, s2, sst);
    }
  }

  // ---- store: acc^T[h][owner row] -> out[owner row][h].  A lane holds 8 bytes in each of 16 places of its
  // row; the rounded rows go through this wave's own LDS region (the stages are free after the last block's
  // barrier), 16-byte chunks XORed with the row, and leave with 16-byte stores that cover whole rows.
  {
    constexpr int OCPR = HP / 8;  // 16-byte chunks per output row
    static_assert(4 * 32 * ROWB <= 4 * TILE, "the output rows are staged in the tile stages");
    char* region = lds + wave * (32 * ROWB);
    auto store = [&](void* out, const floatx16 (&acc)[HT], float mul) {
      static_for<HT>([&](auto HTI) {
        constexpr int ht = decltype(HTI)::value;
        const floatx16 o = acc[ht];
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
          union { T e[4]; u32x2 w; } r;
          r.e[0] = (T)(o[4 * qd + 0] * mul);
          r.e[1] = (T)(o[4 * qd + 1] * mul);
          r.e[2] = (T)(o[4 * qd + 2] * mul);
          r.e[3] = (T)(o[4 * qd + 3] * mul);
          const int chunk = (4 * ht + qd) ^ (l32 & (OCPR - 1));
          *reinterpret_cast<u32x2*>(region + l32 * ROWB + (chunk << 4) + g * 8) = r.w;
        }
      });
      constexpr int RPI = 64 / OCPR;  // rows per store instruction
      const int c = lane % OCPR;
#pragma unroll
      for (int it = 0; it < 32 / RPI; ++it) {
        const int row = it * RPI + lane / OCPR;
        const u32x4 v = *reinterpret_cast<const u32x4*>(region + row * ROWB + ((c ^ (row & (OCPR - 1))) << 4));
        if (wo0 + row < n_own && c * 8 < H)  // H % 8 == 0: a chunk lies inside the row or outside as a whole
          *reinterpret_cast<u32x4*>(reinterpret_cast<T*>(out) + ((int64_t)unit * n_own + wo0 + row) * H + c * 8) = v;
      }
    };
    if constexpr (DS) store(p.out1, acc1, p.scale);
    if constexpr (PV) store(p.out2, acc2, 1.0f);
  }
}

// Keys own, dS from memory: dK = scale dS^T Q, and with PV also dV = P^T dO, whose P it forms again from S.
// Forming dS here takes two products (S and dP) for the one that uses it, and the registers of a second owner operand,
// without which both accumulators fit at two waves per SIMD.  The queries-own pass has dS at hand; it costs a write and a
// read of 2 bytes per score: [8,32,2048,128] causal bf16 1309 -> 1075 us (in one trace of both forms dQ 482 -> 540, dK and dV
// 488 + 354 -> 490), without a mask 2145 -> 1775; 600 x 300 causal heads of 128 95 -> 72; 64 x 2048 heads of 256 953 -> 703.
// At heads of 64 the traffic weighs twice as much and dK and dV share their products anyway: 180 -> 194 us, not used.
// What bounds the two launches: by the counters of a first call the matrix pipe is busy 42 and 48 % of the cycles, the vector
// port 42 and 27 %, a third of the waves' time is waits for an instruction to issue, and memory moves 3.9 and 4.2 TB/s: no
// unit alone, at the clock that the package's power limit leaves (1.9 GHz in that call, 1.75 over a second of them).
// A work-group owns 128 keys and walks the queries in blocks of 32 through three LDS stages (two blocks ahead, 75 KiB, two
// work-groups per CU).
constexpr int SBS = 32;
template <int HP, bool PV> struct SavedLds {
  static constexpr int TILE = SBS * HP * 2, DSB = BO * SBS * 2, STAT = PV ? 4 * 256 : 0;
  static constexpr int STAGE = (PV ? 2 : 1) * TILE + DSB + STAT, ALL = 3 * STAGE;
};
template <typename T, int HC, bool CAUSAL, bool PV>
__device__ __forceinline__ void bwd_saved_pass(const SavedParams& p, char* lds, int block_id) {
  typedef typename Elem<T>::vec8 V8;
  constexpr int HP = padded(HC);
  typedef SavedLds<HP, PV> L;
  constexpr int NW = 4;
  constexpr int ROWB = HP * 2, CPR = ROWB / 16, RPL = 1024 / ROWB, LROWS = NW * RPL;
  constexpr int NL = L::TILE / 1024 / NW;  // loads per wave per tile
  constexpr int KV = (LROWS % 16 == 0) ? 1 : 2;
  constexpr int KS = HC / 16, HT = HC / 32;
  constexpr int LOADS = NL * (PV ? 2 : 1) + 2 + (PV ? 1 : 0);  // loads per wave per block
  static_assert(NL >= 1 && L::DSB == NW * 2 * 1024, "tile / wave split");
  static_assert(!PV || BO * ROWB <= L::ALL, "the owner rows are staged in the stages");
  static_assert(NW * 32 * ROWB <= L::ALL, "and so are the output rows");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, l32 = lane & 31;
  auto swz = [](int row) {
    return CPR >= 16 ? (((row & 3) << 2) | ((row >> 2) & 3)) : ((((row >> 1) & 1) << 2) | ((row >> 2) & 3));
  };
  const int wg = (block_id % 8) * p.per_xcd + block_id / 8;
  if (wg >= p.total || block_id >= 8 * p.per_xcd) return;
  const int UG = p.ug;
  const int ublk = wg / (UG * p.nob), r = wg % (UG * p.nob);
  const int gb = min(UG, p.total / p.nob - ublk * UG);
  const int unit = ublk * UG + r % gb;
  const int ob = r / gb;
  const int o0 = ob * BO;
  const int H = p.H;
  const int wo0 = o0 + wave * 32, orow = wo0 + l32;
  const T* Q = reinterpret_cast<const T*>(p.strm1) + (int64_t)unit * p.F * H;
  const T* dO = reinterpret_cast<const T*>(p.strm2) + (int64_t)unit * p.F * H;
  const T* K = reinterpret_cast<const T*>(p.own1) + (int64_t)unit * p.T * H;
  const float* lse = p.lse + (int64_t)unit * p.F;
  const int nkb = ds_key_blocks(p.T);
  const char* const ds_unit = p.ds + (int64_t)DS_TILE * unit * ds_before((p.F + BO - 1) / BO, nkb, CAUSAL);

  const int lrow = wave * RPL + lane / CPR;
  uint32_t koff[KV];
#pragma unroll
  for (int v = 0; v < KV; ++v) {
    const int chunk = (lane % CPR) ^ swz(lrow + v * LROWS);
    koff[v] = chunk * 8 < H ? (uint32_t)((lrow * H + chunk * 8) * 2) : kOob;
  }
  const uint32_t lstride = (uint32_t)(LROWS * H * 2);
  // 32 rows from t0 on; rows past n_rows come as zeros.
  auto issue_rows = [&](const T* base, int t0, char* __restrict__ tile, int n_rows) {
    const int rows_left = n_rows - t0;
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(base + (int64_t)t0 * H, 0x7fffffffu);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const uint32_t off = lrow + i * LROWS < rows_left ? koff[i % KV] : kOob;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void_ptr)(tile + (i * NW + wave) * 1024), 16, off, i * lstride, 0, 0);
    }
  };
  const int b0 = CAUSAL ? o0 / SBS : 0, b1 = (p.F + SBS - 1) / SBS;
  // Everything of query block it; past the last block nothing is read, and the number of loads is the same.
  auto issue_block = [&](int it, char* __restrict__ st) {
    issue_rows(Q, it * SBS, st, p.F);
    if constexpr (PV) issue_rows(dO, it * SBS, st + L::TILE, p.F);
    char* const d = st + (PV ? 2 : 1) * L::TILE;
    const int rb = it / (BO / SBS);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(
        ds_unit + (int64_t)DS_TILE * (ds_before(rb, nkb, CAUSAL) + (int64_t)(it % (BO / SBS)) * ds_width(rb, nkb, CAUSAL) + ob * (BO / BS)),
        (uint32_t)L::DSB);
    // (Past the end the lanes' offsets turn the loads off, not a buffer of no bytes: they are out of range whether the check adds
    // the scalar offset, leaves it out or takes it from the buffer's size, which must then not be the smaller of the two.)
    const uint32_t off = it < b1 ? (uint32_t)(lane * 16) : kOob;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void_ptr)(d + (i * NW + wave) * 1024), 16, off, (i * NW + wave) * 1024, 0,
                                               kNonTemporal);
    if constexpr (PV) {  // each wave its own copy: 32 floats (the other lanes' 32 are not used)
      const __amdgpu_buffer_rsrc_t rl = make_rsrc(lse, (uint32_t)p.F * 4);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rl, (lds_void_ptr)(d + L::DSB + wave * 256), 4, (uint32_t)((it * SBS + lane) * 4), 0, 0, 0);
    }
  };

  int kbase[KS];  // row fragment s: tile row l%32, logical chunk 2 s + g
#pragma unroll
  for (int s = 0; s < KS; ++s) kbase[s] = l32 * ROWB + (((2 * s + g) ^ swz(l32)) << 4);
  int tbase[HT][2];  // transposed fragments, as in bwd_pass
  const int pl = lane & 15;
#pragma unroll
  for (int ht = 0; ht < HT; ++ht) {
    const int col = 32 * ht + ((lane >> 4) & 1) * 16 + 4 * (pl & 3);
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
      const int row = 4 * g + (pl >> 2) + 8 * h2;
      tbase[ht][h2] = row * ROWB + (((col >> 3) ^ swz(row)) << 4) + (col & 7) * 2;
    }
  }
  // dS fragment (16 queries u, this wave's 32 keys): 4 queries x 16 keys per 16 lanes; + u * 1024, + 512 for the second read.
  const int dbase = (wave >> 1) * DS_TILE + (wave & 1) * 2048 + g * 256 + ((lane >> 4) & 1) * 128 + (pl & 1) * 64 +
                    (pl >> 2) * 16 + ((pl >> 1) & 1) * 8;
  auto tr_read = [](const char* __restrict__ lo_at, const char* __restrict__ hi_at) -> V8 {
    typedef short4v __attribute__((address_space(3))) * lds_ptr;
    const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)lo_at));
    const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)hi_at));
    return __builtin_bit_cast(V8, u32x4{lo[0], lo[1], hi[0], hi[1]});
  };

  V8 of[PV ? KS : 1];
  if constexpr (PV) {
#pragma unroll
    for (int i = 0; i < BO / SBS; ++i) issue_rows(K, o0 + i * SBS, lds + i * L::TILE, p.T);
    __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int s = 0; s < KS; ++s) of[s] = __builtin_bit_cast(V8, *reinterpret_cast<const u32x4*>(lds + wave * L::TILE + kbase[s]));
    __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));
    __builtin_amdgcn_s_barrier();
  }

  floatx16 acc1[HT], acc2[PV ? HT : 1];
#pragma unroll
  for (int i = 0; i < HT; ++i) acc1[i] = zero16();
#pragma unroll
  for (int i = 0; i < (PV ? HT : 1); ++i) acc2[i] = zero16();
  const float scale2 = p.scale * kLog2e;

  auto block = [&](int it, const char* __restrict__ st, char* __restrict__ next) {
    const int t0 = it * SBS;
    issue_block(it + 2, next);
    const char* const qt = st;
    const char* const ot = st + L::TILE;
    const char* const dt = st + (PV ? 2 : 1) * L::TILE;
    if (!CAUSAL || t0 + SBS - 1 >= wo0) {  // (all of a wave's keys lie past these queries: nothing to add)
      floatx16 sc;
      if constexpr (PV) {
        sc = zero16();
#pragma unroll
        for (int s = 0; s < KS; ++s)
          sc = Elem<T>::mfma(__builtin_bit_cast(V8, *reinterpret_cast<const u32x4*>(qt + kbase[s])), of[s], sc);
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const V8 df = tr_read(dt + dbase + u * 1024, dt + dbase + u * 1024 + 512);
#pragma unroll
        for (int ht = 0; ht < HT; ++ht)
          acc1[ht] = Elem<T>::mfma(tr_read(qt + u * 16 * ROWB + tbase[ht][0], qt + u * 16 * ROWB + tbase[ht][1]), df, acc1[ht]);
      }
      if constexpr (PV) {
        V8 pf[2];
        auto probs = [&](auto MASKED_T) {
#pragma unroll
          for (int qd = 0; qd < 4; ++qd) {
            const floatx4 l2 = *reinterpret_cast<const floatx4*>(dt + L::DSB + wave * 256 + (8 * qd + 4 * g) * 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              float arg = __builtin_fmaf(sc[4 * qd + e], scale2, -l2[e]);
              if constexpr (decltype(MASKED_T)::value) {
                const int q = t0 + 8 * qd + 4 * g + e;
                arg = (q >= p.F || (CAUSAL && orow > q)) ? -INFINITY : arg;
              }
              pf[qd >> 1][4 * (qd & 1) + e] = (T)__builtin_amdgcn_exp2f(arg);
            }
          }
        };
        if (t0 + SBS > p.F || (CAUSAL && wo0 + 31 > t0)) probs(std::true_type{});
        else probs(std::false_type{});
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int ht = 0; ht < HT; ++ht)
            acc2[ht] = Elem<T>::mfma(tr_read(ot + u * 16 * ROWB + tbase[ht][0], ot + u * 16 * ROWB + tbase[ht][1]), pf[u], acc2[ht]);
      }
    }
    // The next block's loads have landed; those of the one after it may be in flight.
    __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(LOADS));
    __builtin_amdgcn_s_barrier();
  };

  if (b0 < b1) {
    char* const st0 = lds;
    char* const st1 = lds + L::STAGE;
    char* const st2 = lds + 2 * L::STAGE;
    issue_block(b0, st0);
    issue_block(b0 + 1, st1);
    __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(LOADS));
    __builtin_amdgcn_s_barrier();
    for (int it = b0; it < b1; it += 3) {
      block(it, st0, st2);
      if (it + 1 < b1) block(it + 1, st1, st0);
      if (it + 2 < b1) block(it + 2, st2, st1);
    }
    __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));  // (the loads past the end: zeros for the stages)
    __builtin_amdgcn_s_barrier();
  }

  // ---- store, as in bwd_pass
  constexpr int OCPR = HP / 8;
  char* const region = lds + wave * (32 * ROWB);
  auto store = [&](void* out, const floatx16 (&acc)[HT], float mul) {
    static_for<HT>([&](auto HTI) {
      constexpr int ht = decltype(HTI)::value;
      const floatx16 o = acc[ht];
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        union { T e[4]; u32x2 w; } v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v.e[e] = (T)(o[4 * qd + e] * mul);
        *reinterpret_cast<u32x2*>(region + l32 * ROWB + (((4 * ht + qd) ^ (l32 & (OCPR - 1))) << 4) + g * 8) = v.w;
      }
    });
    constexpr int RPI = 64 / OCPR;
    const int c = lane % OCPR;
#pragma unroll
    for (int i = 0; i < 32 / RPI; ++i) {
      const int row = i * RPI + lane / OCPR;
      const u32x4 v = *reinterpret_cast<const u32x4*>(region + row * ROWB + ((c ^ (row & (OCPR - 1))) << 4));
      if (wo0 + row < p.T && c * 8 < H)
        *reinterpret_cast<u32x4*>(reinterpret_cast<T*>(out) + ((int64_t)unit * p.T + wo0 + row) * H + c * 8) = v;
    }
  };
  store(p.out1, acc1, p.scale);
  if constexpr (PV) store(p.out2, acc2, 1.0f);
}

template <typename T, int HC, bool CAUSAL, bool PV>
__global__ __launch_bounds__(256, 2) void fmha_bwd_saved_kernel(SavedParams p) {
  __shared__ __attribute__((aligned(1024))) char lds[SavedLds<padded(HC), PV>::ALL];
  bwd_saved_pass<T, HC, CAUSAL, PV>(p, lds, (int)blockIdx.x);
}

template <typename T, int HC, bool OWNER_K, bool CAUSAL, bool DS, bool PV, bool BIAS, bool SAVE_DS>
__global__ __launch_bounds__(256, (HC <= 128 && !BIAS && !(DS && PV && HC > 64)) ? 2 : 1) void fmha_bwd_kernel(std::conditional_t<SAVE_DS, SavedParams, KParams> p) {
  __shared__ __attribute__((aligned(1024))) char lds[bwd_lds_bytes(padded(HC))];
  bwd_pass<T, HC, OWNER_K, CAUSAL, DS, PV, BIAS, false, SAVE_DS>(p, lds, (int)blockIdx.x);
}

// All passes in one grid, a row of it each, on statistics formed before: for problems of which a single pass leaves the
// device idle.  What bounds those is the walk of one work-group over the streamed rows (2 us per 64 rows, one wave per
// SIMD), once per launch: [2,7,463,128] causal took three of them.
template <typename T, int HC, bool CAUSAL>
__global__ __launch_bounds__(256, HC <= 128 ? 2 : 1) void fmha_bwd_small_kernel(KParams dq, KParams dk, KParams dv) {
  __shared__ __attribute__((aligned(1024))) char lds[bwd_lds_bytes(padded(HC))];
  const int block = (int)blockIdx.x;
  if (blockIdx.y == 0) bwd_pass<T, HC, false, CAUSAL, true, false, false, true, false>(dq, lds, block);
  else if constexpr (HC <= 64) bwd_pass<T, HC, true, CAUSAL, true, true, false, true, false>(dk, lds, block);
  else if (blockIdx.y == 1) bwd_pass<T, HC, true, CAUSAL, true, false, false, true, false>(dk, lds, block);
  else bwd_pass<T, HC, true, CAUSAL, false, true, false, true, false>(dv, lds, block);
}

void split(KParams& p, int n_own, uint64_t units) {
  p.nob = (n_own + BO - 1) / BO;
  p.total = (int)(units * p.nob);
  p.per_xcd = (p.total + 7) / 8;
  p.ug = std::max(4, (64 + p.nob - 1) / p.nob);  // enough units to fill an XCD's slots with one round
}

template <typename T, int HC, bool OWNER_K, bool DS, bool PV>
void launch_pass(KParams p, uint64_t units, bool causal, hipStream_t st) {
  split(p, OWNER_K ? p.T : p.F, units);
  const dim3 grid((unsigned)(p.per_xcd * 8)), block(256);
  if (p.bias) {
    if (causal) hipLaunchKernelGGL((fmha_bwd_kernel<T, HC, OWNER_K, true, DS, PV, true, false>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((fmha_bwd_kernel<T, HC, OWNER_K, false, DS, PV, true, false>), grid, block, 0, st, p);
  } else {
    if (causal) hipLaunchKernelGGL((fmha_bwd_kernel<T, HC, OWNER_K, true, DS, PV, false, false>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((fmha_bwd_kernel<T, HC, OWNER_K, false, DS, PV, false, false>), grid, block, 0, st, p);
  }
}

// The same pass from unit u0 on (no bias); `owner_k` says which of q / o / dO and k / v are the owners.
SavedParams at_unit(const KParams& from, char* ds, uint64_t u0, bool owner_k) {
  SavedParams p{from, ds};
  const uint64_t rows_q = u0 * p.F, q = rows_q * p.H * 2, k = u0 * p.T * p.H * 2;
  auto at = [](const void* v, uint64_t bytes) { return static_cast<const void*>(static_cast<const char*>(v) + bytes); };
  auto to = [](void* v, uint64_t bytes) { return v ? static_cast<void*>(static_cast<char*>(v) + bytes) : nullptr; };
  const uint64_t own = owner_k ? k : q, strm = owner_k ? q : k;
  p.own1 = at(p.own1, own); p.own2 = at(p.own2, own); p.strm1 = at(p.strm1, strm); p.strm2 = at(p.strm2, strm);
  p.o = at(p.o, q); p.lse += rows_q; p.dsum += rows_q; p.lse_fwd += rows_q;
  p.out1 = to(p.out1, own); p.out2 = to(p.out2, own);
  return p;
}

// dQ and dS (kept), then dK and dV from it; with heads of more than 128 dV has its own pass, as its accumulators need.
template <typename T, int HC, bool CAUSAL>
void launch_saved(SavedParams p, SavedParams kv, uint64_t units, hipStream_t st) {
  split(p, p.F, units);
  split(kv, kv.T, units);
  const dim3 block(256);
  hipLaunchKernelGGL((fmha_bwd_kernel<T, HC, false, CAUSAL, true, false, false, true>), dim3((unsigned)(p.per_xcd * 8)), block, 0, st, p);
  hipLaunchKernelGGL((fmha_bwd_saved_kernel<T, HC, CAUSAL, (HC <= 128)>), dim3((unsigned)(kv.per_xcd * 8)), block, 0, st, kv);
  if constexpr (HC > 128) launch_pass<T, HC, true, false, true>(kv, units, CAUSAL, st);
}

template <typename T, int HC>
void launch_both(const fmha_bwd_fused::Args& a, uint64_t units, hipStream_t st) {
  KParams p;
  p.lse = a.lse; p.dsum = a.dsum; p.o = a.o; p.lse_fwd = a.lse_fwd; p.H = a.H; p.F = a.F; p.T = a.T; p.scale = a.scale;
  p.bias = a.bias;
  p.bias_vec = a.bias && a.T % 4 == 0 && xmk::aligned(a.bias, 8);
  p.nob = p.total = p.per_xcd = 0;
  p.own1 = a.q; p.own2 = a.d_o; p.strm1 = a.k; p.strm2 = a.v; p.out1 = a.dq; p.out2 = nullptr;
  KParams k = p;
  k.own1 = a.k; k.own2 = a.v; k.strm1 = a.q; k.strm2 = a.d_o; k.out1 = a.dk; k.out2 = a.dv;
  if constexpr (HC > 64) if (a.ds) {
    char* const ds = static_cast<char*>(a.ds);
    for (uint64_t u0 = 0; u0 < units; u0 += a.ds_units) {
      const uint64_t n = std::min<uint64_t>(a.ds_units, units - u0);
      if (a.causal) launch_saved<T, HC, true>(at_unit(p, ds, u0, false), at_unit(k, ds, u0, true), n, st);
      else launch_saved<T, HC, false>(at_unit(p, ds, u0, false), at_unit(k, ds, u0, true), n, st);
    }
    return;
  }
  if (a.stats_ready) {
    split(p, a.F, units);
    split(k, a.T, units);
    const dim3 grid((unsigned)(std::max(p.per_xcd, k.per_xcd) * 8), HC <= 64 ? 2 : 3), block(256);
    if (a.causal) hipLaunchKernelGGL((fmha_bwd_small_kernel<T, HC, true>), grid, block, 0, st, p, k, k);
    else hipLaunchKernelGGL((fmha_bwd_small_kernel<T, HC, false>), grid, block, 0, st, p, k, k);
    return;
  }
  // owner = queries first: dQ, and the per-row statistics the other launches read
  launch_pass<T, HC, false, true, false>(p, units, a.causal, st);
  // owner = keys: dK, then dV
  // One pass for both where the two accumulators fit beside everything else (S is then computed once for the
  // two): head size <= 64 (S = 4096, H = 64 causal: 0.69 -> 0.57 ms), and head size <= 128 with a bias, whose
  // kernels run one wave per SIMD anyway (6.2 -> 5.3 ms).  Without a bias the merged H = 128 pass would have to
  // give up the second wave per SIMD and comes out 2-4 % slower; at H = 256 it spills.
  if constexpr (HC <= 128) if (HC <= 64 || a.bias) {
    launch_pass<T, HC, true, true, true>(k, units, a.causal, st);
    return;
  }
  if constexpr (HC > 64) {
    launch_pass<T, HC, true, true, false>(k, units, a.causal, st);
    launch_pass<T, HC, true, false, true>(k, units, a.causal, st);
  }
}

}  // namespace

namespace fmha_bwd_fused {

bool eligible(const Args& a, uint64_t units) {
  return a.H <= 256 && a.H % 8 == 0 && units * ((uint64_t)((a.F > a.T ? a.F : a.T) + BO - 1) / BO) < 0x7fffffffull &&
         (uint64_t)a.F * a.H * 2 < kOob && (uint64_t)a.T * a.H * 2 < kOob &&
         (!a.bias || (uint64_t)a.F * a.T * 2 < kOob);
}

// One grid (plus a launch for the statistics) against a launch per pass, causal bf16: 14 units of 463 rows, heads of 128,
// 56 -> 26 us; 4 x 4096 336 -> 155; 16 x 2048 183 -> 116; heads of 64, 32 x 1024 51 -> 39; heads of 256, 14 x 463
// 121 -> 48.  Up to 384 work-groups per pass all that was timed gained 10 % or more, 512 still 2 - 18 % on 512 rows and
// more; 512 of 64 or 128 rows lost 5 % (23 -> 24 us), 256 x 128 with heads of 256 2 %.  Kernels with a bias run one
// wave per SIMD and hold other accumulators; they keep their launches.
bool one_grid(const Args& a, uint64_t units) {
  const uint64_t rows = (uint64_t)std::max(a.F, a.T), groups = units * ((rows + BO - 1) / BO);
  const uint64_t most = rows >= 512 ? 512 : (a.H > 128 && rows <= 128) ? 128 : 384;
  return !a.bias && groups <= most;
}

// All units in one part run with fewer launches than without dS; what a part of them loses is its last, partly empty
// rounds of 512 work-groups: 896 per part (32 x 16384, 7 units at a time) 8.2 -> 10.9 ms, 1408 (64 x 8192) 4.19 -> 4.02.
// The one grid of a small problem fills the device with the work-groups of all passes; with dS kept each pass has to by
// itself.  One grid / dS kept, us, two work-groups per CU: 512 groups, 32 x 2048, causal 195 / 179, no mask 291 / 236; 384,
// 24 x 2048, 145 / 150 and 235 / 197; 352, 352 x 180, 34.6 / 32.3; 320, 10 x 4096, 278 / 264, but 269 x 61 causal 21.4 / 23.9,
// 277 x 46 20.2 / 22.1, 35 x 1014 79 / 87.  Heads of more than 128: no mask 272 groups of 2154 353 / 418, 302 of 225 111 / 118,
// 348 of 471 5 % faster with it; causal level at 256.  And where queries or keys are few, so is the work of one pass: 86 x 302
// queries and 77 keys 26.0 / 30.9, 48 x 54 and 884 29.9 / 39.2, 69 x 125 and 583, heads of 256, 72 / 98 (up to 160 rows of
// such heads: level).  Of 858 drawn sizes 4 lose more than 2 % by this rule, the worst 3 %; with 256 work-groups of the
// longer side as the rule 49 did, up to 48 %.
uint64_t saved_units(const Args& a, uint64_t units, uint64_t bytes) {
  constexpr uint64_t kMost = (uint64_t)2 << 30, kPartGroups = 1280;
  auto groups = [&](uint64_t rows) { return units * ((rows + BO - 1) / BO); };
  const uint64_t rows = (uint64_t)std::max(a.F, a.T), per_unit = (rows + BO - 1) / BO;
  if (a.bias || a.H <= 64 || groups(rows) < 256) return 0;
  if (one_grid(a, units) && (a.H <= 128 || rows > 160)) {
    if (groups(rows) < (a.H > 128 ? a.causal ? 256u : 336u : a.causal && rows > 1024 ? 385u : 352u)) return 0;
    if (groups((uint64_t)std::min(a.F, a.T)) < 128) return 0;
  }
  const uint64_t fit = std::min(bytes, kMost) / saved_bytes(a, 1);
  if (fit >= units) return units;
  if (fit == 0) return 0;
  const uint64_t parts = (units + fit - 1) / fit, each = (units + parts - 1) / parts;
  return each * per_unit >= kPartGroups ? each : 0;
}

size_t saved_bytes(const Args& a, uint64_t units) { return units * ds_unit_bytes(a.F, a.T, a.causal); }

void launch(const Args& a, uint64_t units, bool bf16, hipStream_t st) {
  // The products run over the head's own steps of 16 and tiles of 32; of 96 and 160 instead of 128 and 256 (us, both in one
  // grid): 13 causal heads of 524 x 80 26.9 -> 23.0, 36 of 753 x 80 53.7 -> 42.1, 16 of 1024 x 160 127 -> 91, 8 of 256 x 160 26 -> 20.
  if (bf16) {
    if (a.H <= 64) launch_both<__bf16, 64>(a, units, st);
    else if (a.H <= 96) launch_both<__bf16, 96>(a, units, st);
    else if (a.H <= 128) launch_both<__bf16, 128>(a, units, st);
    else if (a.H <= 160) launch_both<__bf16, 160>(a, units, st);
    else launch_both<__bf16, 256>(a, units, st);
  } else {
    if (a.H <= 64) launch_both<_Float16, 64>(a, units, st);
    else if (a.H <= 96) launch_both<_Float16, 96>(a, units, st);
    else if (a.H <= 128) launch_both<_Float16, 128>(a, units, st);
    else if (a.H <= 160) launch_both<_Float16, 160>(a, units, st);
    else launch_both<_Float16, 256>(a, units, st);
  }
}

}  // namespace fmha_bwd_fused
