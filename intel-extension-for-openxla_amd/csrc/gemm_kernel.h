// MFMA GEMM kernel and its launch templates (included by gemm.hip for the host API and by the
// gemm_inst_*.hip units, each of which instantiates one (element type, output type) pair so
// that the instantiations compile in parallel).
#pragma once
#include <hip/hip_bf16.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <utility>

#include "common.h"
#include "tile_order.h"

namespace gemm_impl {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));


enum : int { ACT_NONE = 0, ACT_RELU = 1, ACT_GELU = 2 };

struct GemmParams {
  // What a work-group needs for its first loads (request_first_args).
  const void* a;
  const void* b;
  int64_t lda, ldb;             // elements between stored rows
  int64_t sa, sb;               // batch strides, elements
  int M, N, K;
  int kslice;                   // K slice of one grid member (a multiple of the K step), 0 when K is not split
  TileOrder order;
  // The rest.
  int tiles_m, tiles_n;
  void* out;
  const void* c;
  const void* bias;
  int64_t ldc, sc;
  float alpha, beta;
  int act;
  // Shared-lhs multi-output form (three GEMMs with one A): batch member z > 0 writes to
  // out_alt[z - 1] instead of out + z * sc and reads bias + z * sbias.  Null when unused.
  void* out_alt[2];
  int64_t sbias;
  // int8 kernel only: elements per load that the alignment of each operand's pointer, leading dimension, batch
  // stride and row length allows.
  int vec_a, vec_b;
  // Kernels that take any alignment: some row of an operand does not start on a 16-byte boundary.
  bool misaligned;
};

// Asks for the arguments in front of the first loads at once: where their uses are spread over the prologue, the compiler asks
// for them there, and every cache line of them is a round trip to memory of its own (the smallest launches 0.1 to 0.3 us).
__device__ __forceinline__ void request_first_args(const GemmParams& p) {
  const TileOrder& o = p.order;
  asm volatile("" ::"s"(p.a), "s"(p.b), "s"(p.lda), "s"(p.ldb), "s"(p.sa), "s"(p.sb), "s"(p.M), "s"(p.N), "s"(p.K), "s"(p.kslice),
               "s"(o.xcd_step), "s"(o.rest), "s"(o.round_step), "s"(o.group), "s"(o.inv_group), "s"(o.last_group), "s"(o.last_rows),
               "s"(o.inv_last), "s"(o.shift));
}

__device__ __forceinline__ float gelu_tanh(float x) {
  // 0.5 x (1 + tanh(u)) = x * sigmoid(2u) = x / (1 + exp(-2u)), u = sqrt(2/pi)(x + 0.044715 x^3)
  const float u = 0.7978845608028654f * (x + 0.044715f * x * x * x);
  return x / (1.0f + __expf(-2.0f * u));
}
// The same for results of 16 bits, which do not show the reciprocal's last bit (error against float64 the same to seven digits):
// eight instructions, where the division alone takes ten.  A large tile has one wave per SIMD and nothing beside its epilogue:
// 1659 x 11592 x 120 47.4 -> 36.8 us, 6870 x 3856 x 936 89.6 -> 78.7, 1023 x 5003 x 2047 with scratch 42.9 -> 38.5.
__device__ __forceinline__ float gelu_tanh_16(float x) {
  constexpr float k1 = -2.0f * 0.7978845608028654f * 1.4426950408889634f;
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * __builtin_fmaf(0.044715f * k1, x * x, k1)));
}

__device__ __forceinline__ float apply_act(float v, int act) {
  if (act == ACT_RELU) return fmaxf(v, 0.0f);
  if (act == ACT_GELU) return gelu_tanh(v);
  return v;
}

template <typename T> struct Elem;
template <> struct Elem<__bf16> {
  typedef bf16x8 vec8;
  static __device__ __forceinline__ floatx16 mfma(vec8 a, vec8 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ float to_f32(__bf16 v) { return (float)v; }
  static __device__ __forceinline__ uint16_t from_f32(float v) {
    __bf16 h = (__bf16)v;
    return __builtin_bit_cast(uint16_t, h);
  }
};
template <> struct Elem<_Float16> {
  typedef f16x8 vec8;
  static __device__ __forceinline__ floatx16 mfma(vec8 a, vec8 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ float to_f32(_Float16 v) { return (float)v; }
  static __device__ __forceinline__ uint16_t from_f32(float v) {
    _Float16 h = (_Float16)v;
    return __builtin_bit_cast(uint16_t, h);
  }
};

// Compile-time loop: f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>).  Used where
// an index into a register array must be a constant no matter what the unroller decides.
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(static_cast<F&&>(f), std::make_integer_sequence<int, N>{});
}

__device__ __forceinline__ floatx16 zero16() {
  return floatx16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
}

// Buffer descriptor over [base, base + 2 GiB): loads whose byte offset is >= 2^31 (the
// sentinel kOob) return zero, which is how out-of-range rows / k are zero-filled.
constexpr uint32_t kOob = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)kOob, 0x00020000);
}

typedef __attribute__((address_space(3))) void* lds_void_ptr;

// XOR applied to the 16-byte chunk index inside an LDS row, chosen so that the lanes the LDS serves
// together touch different banks (256 bytes of banks).
//   KC, BK = 64: rows of 128 bytes (8 chunks); KC, BK = 32: rows of 64 bytes (4 chunks); read with
//       ds_read_b128, 16 lanes = 16 rows of one chunk column.  Two (four) rows share 256 bytes of banks and
//       are apart by their position there, so the XOR counts pairs (quadruples) of rows.
//   MC: rows of ROWS * 2 bytes, read with the LDS transpose loads.  16-bit elements (EB = 2,
//       ds_read_b64_tr_b16): 32 lanes take 64 bytes of each of 4 consecutive k rows, so rows of 256 bytes and
//       more move by whole 64-byte groups, (k & 3) << 2; with 128-byte rows two rows share the banks and
//       (k & 3) << 1 separates the four.  8-bit elements (EB = 1, ds_read_b64_tr_b8): 32 lanes take 32 bytes of
//       each of 8 consecutive k rows, (k & 7) << 1 (rows of 256 bytes and more).  The XOR is even so that 32-byte pairs
//       stay together.
template <bool MC, int ROWS, int BK, int EB = 2>
__device__ __forceinline__ int swz(int row_or_k) {
  if constexpr (!MC) return BK == 64 ? ((row_or_k >> 1) & 7) : ((row_or_k >> 2) & 3);
  else if constexpr (ROWS < 64) return 0;  // four rows of 64 bytes are one sweep of the banks
  else if constexpr (ROWS < 128) return (row_or_k & 3) << 1;  // 8 chunks per row: the XOR stays below 8
  else if constexpr (EB == 1) return (row_or_k & 7) << 1;
  else return (row_or_k & 3) << 2;
}

// One operand tile = BK k x ROWS rows/cols = ROWS * BK * 2 bytes of LDS in both layouts.
// A wave issues NL loads of 1 KiB per K step; load j = i * NWAVES + wave (i = 0..NL-1) fills
// LDS bytes [1024 j, 1024 j + 1024).  The swizzle is chosen so that a lane fetches the same
// chunk column in every load: its global byte offset is voff + i * sstride, with voff in one
// VGPR and the per-load part in the instruction's scalar offset.  Row/column validity is
// kept as one lane mask per load (scalar registers).
template <bool MC, int ROWS, int BK, int NWAVES, int EB = 2>
struct Loader {
  static constexpr int RB = MC ? ROWS * 2 : BK * 2;  // LDS row, bytes
  static constexpr int CPR = RB / 16;                // chunks per LDS row
  static constexpr int RPL = 1024 / RB;              // LDS rows per load
  static constexpr int NL = ROWS * BK * 2 / 1024 / NWAVES;
  static constexpr int LSTRIDE = NWAVES * RPL;       // LDS rows between consecutive loads of a wave
  static_assert(NL >= 1, "tile too small for this many waves");
  static_assert(LSTRIDE % 16 == 0 || (LSTRIDE % 8 == 0 && (MC || BK == 32)), "swizzle must repeat from load to load");
  uint32_t voff;     // byte offset of this lane's chunk in load 0, from the tile origin
  uint32_t sstride;  // bytes between consecutive loads of this wave (uniform)
  int kin0;          // k (inside the K step) of this lane's chunk in load 0
  bool ok[NL];       // this lane's row / column exists
  uint32_t okoff[NL];  // ok[i] ? voff : kOob -- the offset of load i in a K step that lies fully inside K

  __device__ __forceinline__ void init(int64_t ld, int valid, int wave, int lane) {
    const int lrow = wave * RPL + lane / CPR;  // LDS row in load 0: operand row (KC) or k (MC)
    const int chunk = (lane % CPR) ^ swz<MC, ROWS, BK, EB>(lrow);
    voff = (uint32_t)(((int64_t)lrow * ld + chunk * 8) * 2);
    sstride = (uint32_t)(LSTRIDE * ld * 2);
    if constexpr (!MC) {
      kin0 = chunk * 8;
#pragma unroll
      for (int i = 0; i < NL; ++i) ok[i] = lrow + i * LSTRIDE < valid;
    } else {
      kin0 = lrow;
#pragma unroll
      for (int i = 0; i < NL; ++i) ok[i] = chunk * 8 < valid;
    }
#pragma unroll
    for (int i = 0; i < NL; ++i) okoff[i] = ok[i] ? voff : kOob;
  }
  // Issues load i.  base: address of the tile origin for this K step; kleft: k of the step that
  // exist (<= 0 past the end of K: every lane is then out of range and the load writes zeros).
  // CHECK_K = false: the caller knows that the whole K step exists (kleft >= BK).
  template <bool CHECK_K = true>
  __device__ __forceinline__ void issue_one(int i, __amdgpu_buffer_rsrc_t rsrc, int kleft, char* lds_tile,
                                            int wave) const {
    const int k = MC ? kin0 + i * LSTRIDE : kin0;
    const uint32_t off = CHECK_K ? ((ok[i] && k < kleft) ? voff : kOob) : okoff[i];
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_ptr)(lds_tile + (i * NWAVES + wave) * 1024), 16,
                                             off, i * sstride, 0, 0);
  }
  __device__ __forceinline__ void issue(const void* base, int kleft, char* lds_tile, int wave) const {
    const __amdgpu_buffer_rsrc_t rsrc = make_rsrc(base);
#pragma unroll
    for (int i = 0; i < NL; ++i) issue_one(i, rsrc, kleft, lds_tile, wave);
  }
};

// Per-lane LDS byte offsets of an operand's fragments, computed once.  A fragment of the
// 32-row (or 32-column) slab t for k-step ks (16 k) gives lane l row l%32, k = 16 ks + 8 (l/32)..+7.
//   KC: one 16-byte read at base[ks] + t * 32 * RB          (the XOR depends on ks, not on t)
//   MC: two transpose reads (k .. k+3 and k+4 .. k+7 of one column) at base[t][h] + ks * 16 * RB
//       (the XOR depends on t and h, not on ks)
template <bool MC, int ROWS, int BK, int T>
struct FragAddr {
  static constexpr int KS = BK / 16;
  int base[MC ? T : KS][MC ? 2 : 1];
  __device__ __forceinline__ void init(int row0, int lane) {
    if constexpr (!MC) {
      const int row = row0 + (lane & 31);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        base[ks][0] = row * (BK * 2) + (((ks * 2 + (lane >> 5)) ^ swz<false, ROWS, BK>(row)) << 4);
    } else {
      // Within a 16-lane block, lane p addresses row (kb + p/4), columns (cb + 4 (p%4)) .. +3
      // and receives column cb + p, rows kb .. kb+3.
      const int p = lane & 15;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const int col = row0 + t * 32 + ((lane >> 4) & 1) * 16 + 4 * (p & 3);
        const int chunk = col >> 3, within = (col & 7) * 2;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k = (lane >> 5) * 8 + (p >> 2) + 4 * h;  // + 16 ks, which does not change k & 7
          base[t][h] = k * (ROWS * 2) + ((chunk ^ swz<true, ROWS, BK>(k)) << 4) + within;
        }
      }
    }
  }
  template <typename V8>
  __device__ __forceinline__ V8 read(const char* __restrict__ tile, int t, int ks) const {
    if constexpr (!MC) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(tile + base[ks][0] + t * 32 * (BK * 2));
      return __builtin_bit_cast(V8, v);
    } else {
      typedef short4v __attribute__((address_space(3))) * lds_ptr;
      const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(tile + base[t][0] + ks * 16 * (ROWS * 2)));
      const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(tile + base[t][1] + ks * 16 * (ROWS * 2)));
      u32x4 v;
      v[0] = __builtin_bit_cast(u32x2, lo)[0];
      v[1] = __builtin_bit_cast(u32x2, lo)[1];
      v[2] = __builtin_bit_cast(u32x2, hi)[0];
      v[3] = __builtin_bit_cast(u32x2, hi)[1];
      return __builtin_bit_cast(V8, v);
    }
  }
};

// s_waitcnt immediate (gfx9 encoding) that waits until at most n vector-memory loads are
// outstanding and does not wait on the other counters.
__host__ __device__ constexpr int vmcnt_imm(int n) {
  return (n & 0xf) | ((n >> 4) << 14) | (0x7 << 4) | (0xf << 8);
}

// Epilogue for four consecutive output columns n..n+3 of row m held by one lane.
template <typename T, bool OutF32>
__device__ __forceinline__ void store_quad(const GemmParams& p, floatx4 a, int m, int n,
                                           int64_t coff) {
  if (m >= p.M || n >= p.N) return;
  const int64_t off = coff + (int64_t)m * p.ldc + n;
  const bool full = n + 4 <= p.N;
  float v0 = p.alpha * a[0], v1 = p.alpha * a[1], v2 = p.alpha * a[2], v3 = p.alpha * a[3];
  if (p.c) {  // non-null only when beta != 0
    float c0 = 0.f, c1 = 0.f, c2 = 0.f, c3 = 0.f;
    if constexpr (OutF32) {
      const float* cp = reinterpret_cast<const float*>(p.c) + off;
      c0 = cp[0];
      if (full || n + 1 < p.N) c1 = cp[1];
      if (full || n + 2 < p.N) c2 = cp[2];
      if (full) c3 = cp[3];
    } else {
      const T* cp = reinterpret_cast<const T*>(p.c) + off;
      c0 = Elem<T>::to_f32(cp[0]);
      if (full || n + 1 < p.N) c1 = Elem<T>::to_f32(cp[1]);
      if (full || n + 2 < p.N) c2 = Elem<T>::to_f32(cp[2]);
      if (full) c3 = Elem<T>::to_f32(cp[3]);
    }
    v0 += p.beta * c0; v1 += p.beta * c1; v2 += p.beta * c2; v3 += p.beta * c3;
  }
  if (p.bias) {
    const T* bp = reinterpret_cast<const T*>(p.bias) + n;
    v0 += Elem<T>::to_f32(bp[0]);
    if (full || n + 1 < p.N) v1 += Elem<T>::to_f32(bp[1]);
    if (full || n + 2 < p.N) v2 += Elem<T>::to_f32(bp[2]);
    if (full) v3 += Elem<T>::to_f32(bp[3]);
  }
  v0 = apply_act(v0, p.act); v1 = apply_act(v1, p.act);
  v2 = apply_act(v2, p.act); v3 = apply_act(v3, p.act);
  if constexpr (OutF32) {
    float* op = reinterpret_cast<float*>(p.out) + off;
    if (full && (off % 4 == 0)) {
      *reinterpret_cast<floatx4*>(op) = floatx4{v0, v1, v2, v3};
    } else {
      op[0] = v0;
      if (n + 1 < p.N) op[1] = v1;
      if (n + 2 < p.N) op[2] = v2;
      if (n + 3 < p.N) op[3] = v3;
    }
  } else {
    uint16_t* op = reinterpret_cast<uint16_t*>(p.out) + off;
    const uint16_t h0 = Elem<T>::from_f32(v0), h1 = Elem<T>::from_f32(v1);
    const uint16_t h2 = Elem<T>::from_f32(v2), h3 = Elem<T>::from_f32(v3);
    if (full && (off % 4 == 0)) {
      u32x2 w;
      w[0] = (uint32_t)h0 | ((uint32_t)h1 << 16);
      w[1] = (uint32_t)h2 | ((uint32_t)h3 << 16);
      *reinterpret_cast<u32x2*>(op) = w;
    } else {
      op[0] = h0;
      if (n + 1 < p.N) op[1] = h1;
      if (n + 2 < p.N) op[2] = h2;
      if (n + 3 < p.N) op[3] = h3;
    }
  }
}

// What a tile's products become: out = act(alpha * acc + beta * c + bias) for eight consecutive columns of a row.
// A lane's columns are the same for all its rows, so the bias is fetched once.
template <typename T, bool OutF32>
struct GemmEpilogue {
  const void *c, *bias_vec;  // null when unused
  int64_t ldc, coff;
  float alpha, beta;
  int act;
  float bias[8];
  // bz: batch member
  __device__ __forceinline__ GemmEpilogue(const GemmParams& p, int64_t bz)
      : c(p.c), bias_vec(p.bias ? reinterpret_cast<const T*>(p.bias) + bz * p.sbias : nullptr), ldc(p.ldc), coff(bz * p.sc),
        alpha(p.alpha), beta(p.beta), act(p.act) {}
  // Eight values at any alignment, of which `count` exist (the others repeat the last one: no branches, so that
  // all loads are in flight together).
  template <bool F32>
  static __device__ __forceinline__ void fetch(const void* base, int64_t off, int count, float (&v)[8]) {
    if constexpr (F32) {
      const float* p = reinterpret_cast<const float*>(base) + off;
      if (count >= 8) {
        floatx4 lo, hi;
        __builtin_memcpy(&lo, p, 16);
        __builtin_memcpy(&hi, p + 4, 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) { v[e] = lo[e]; v[4 + e] = hi[e]; }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = p[min(e, count - 1)];
      }
    } else {
      const T* p = reinterpret_cast<const T*>(base) + off;
      if (count >= 8) {
        u32x4 w;
        __builtin_memcpy(&w, p, 16);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = Elem<T>::to_f32(__builtin_bit_cast(T, (uint16_t)(w[e / 2] >> (16 * (e & 1)))));
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = Elem<T>::to_f32(p[min(e, count - 1)]);
      }
    }
  }
  // count: columns from n on that exist (8: all of the lane's).
  __device__ __forceinline__ void columns(int n, int count) {
    if (bias_vec && count > 0) fetch<sizeof(T) == 4>(bias_vec, n, count, bias);
  }
  // U rows at once, rows[u] inside the matrix: every test below is uniform and is made once for them all.
  template <int U>
  __device__ __forceinline__ void apply(float (&v)[U][8], const int (&rows)[U], int n, int count) const {
    if (alpha != 1.0f) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[u][e] *= alpha;
    }
    if (c) {  // non-null only when beta != 0
      float cv[U][8];
#pragma unroll
      for (int u = 0; u < U; ++u) fetch<OutF32>(c, coff + (int64_t)rows[u] * ldc + n, count, cv[u]);
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[u][e] += beta * cv[u][e];
    }
    if (bias_vec) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[u][e] += bias[e];
    }
    if (act == ACT_RELU) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[u][e] = fmaxf(v[u][e], 0.f);
    } else if (act == ACT_GELU) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[u][e] = OutF32 || sizeof(T) == 4 ? gelu_tanh(v[u][e]) : gelu_tanh_16(v[u][e]);
    }
  }
};

// The output of batch member bz (offsets bz * p.sc are added by the caller).
__device__ __forceinline__ void* member_out(const GemmParams& p, int64_t bz) {
  return p.out_alt[0] && bz > 0 ? p.out_alt[bz - 1] : p.out;
}

// Eight results of a row (count of them exist), rounded once, at any alignment: one 16-byte store per 16 bytes.
template <typename T, bool OutF32>
__device__ __forceinline__ void store8(void* out, int64_t off, const float (&v)[8], int count) {
  if constexpr (OutF32) {
    float* p = reinterpret_cast<float*>(out) + off;
    if (count >= 8) {
      __builtin_memcpy(p, v, 32);
    } else {
#pragma unroll
      for (int e = 0; e < 7; ++e)
        if (e < count) p[e] = v[e];
    }
  } else {
    uint16_t* p = reinterpret_cast<uint16_t*>(out) + off;
    uint16_t h[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) h[e] = Elem<T>::from_f32(v[e]);
    if (count >= 8) {
      __builtin_memcpy(p, h, 16);
    } else {
#pragma unroll
      for (int e = 0; e < 7; ++e)
        if (e < count) p[e] = h[e];
    }
  }
}

// Epilogue of a wave's 32 TM x 32 TN part of a tile at (m_base, n_base), which may hang over the M x N matrix.
// acc[i][j][e] is row 32 i + lane % 32, column 32 j + 8 (e / 4) + 4 (lane / 32) + e % 4.  The accumulators go
// through the wave's LDS region (32 x 32 TN floats, 16-byte chunks XORed by the row so that both passes are free
// of bank conflicts) one 32-row slab at a time and come back as eight consecutive columns per lane: the addend,
// the bias and the result move in whole 16-byte pieces (in the accumulator layout a lane has 8 bytes in each of
// 32 rows, and fetched the bias again for every one of them: 5120 x 2048 x 256 with a bias 28.2 us, without 14.5).
template <typename T, bool OutF32, int TM, int TN, class Epilogue>
__device__ __forceinline__ void store_tile(Epilogue& epi, const floatx16 (&acc)[TM][TN], char* region, void* out, int64_t ldc,
                                           int64_t coff, int M, int N, int m_base, int n_base, int lane) {
  constexpr int RBY = TN * 128;             // bytes of a row of the region
  constexpr int XM = TN == 1 ? 7 : 15;      // 16-byte chunks that the XOR moves among
  constexpr int LPR = TN * 4;               // lanes per row when copying out
  constexpr int RPI = 64 / LPR;             // rows per copy step
  const int r1 = lane & 31, h = lane >> 5;
  const int c8 = lane % LPR;
  const int n = n_base + c8 * 8;
  const int count = N - n;
  const bool whole = m_base + 32 * TM <= M && n_base + 32 * TN <= N;
  epi.columns(n, count);
  // The copy-out stays a loop: unrolled, the code outgrew the instruction cache and cost more than the stores
  // (5120 x 2048 x 256 14.5 -> 26 us).
  auto fetch_row = [&](int row, float (&v)[8]) {
    *reinterpret_cast<floatx4*>(v) = *reinterpret_cast<const floatx4*>(region + row * RBY + (((2 * c8) ^ (row & XM)) << 4));
    *reinterpret_cast<floatx4*>(v + 4) = *reinterpret_cast<const floatx4*>(region + row * RBY + (((2 * c8 + 1) ^ (row & XM)) << 4));
  };
  static_for<TM>([&](auto I) {
    static_for<TN>([&](auto J) {
      constexpr int j = decltype(J)::value;
      const floatx16 t = acc[decltype(I)::value][j];
      static_for<4>([&](auto Q) {
        constexpr int qd = decltype(Q)::value;
        *reinterpret_cast<floatx4*>(region + r1 * RBY + (((8 * j + 2 * qd + h) ^ (r1 & XM)) << 4)) =
            floatx4{t[4 * qd], t[4 * qd + 1], t[4 * qd + 2], t[4 * qd + 3]};
      });
    });
    const int m_slab = m_base + decltype(I)::value * 32;
    if (whole) {  // uniform
      constexpr int U = 32 / RPI < 4 ? 32 / RPI : 4;  // rows of a lane in flight together
#pragma unroll 1
      for (int it = 0; it < 32 / RPI; it += U) {
        alignas(16) float v[U][8];
        int rows[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int row = (it + u) * RPI + lane / LPR;
          fetch_row(row, v[u]);
          rows[u] = m_slab + row;
        }
        epi.template apply<U>(v, rows, n, 8);
#pragma unroll
        for (int u = 0; u < U; ++u) store8<T, OutF32>(out, coff + (int64_t)rows[u] * ldc + n, v[u], 8);
      }
    } else {
#pragma unroll 1
      for (int it = 0; it < 32 / RPI; ++it) {
        const int row = it * RPI + lane / LPR;
        if (count > 0 && m_slab + row < M) {
          alignas(16) float v[1][8];
          fetch_row(row, v[0]);
          epi.template apply<1>(v, {m_slab + row}, n, count);
          store8<T, OutF32>(out, coff + (int64_t)(m_slab + row) * ldc + n, v[0], count);
        }
      }
    }
  });
}

// T: element type; OutF32: fp32 output (else T); A_MC / B_MC: operand's free index is
// contiguous; BM x BN tile; WGM x WGN waves; BK: K step (32 or 64); NSTAGE: LDS stages.
template <typename T, bool OutF32, bool A_MC, bool B_MC, int BM, int BN, int WGM, int WGN, int BK, int NSTAGE>
__global__ __launch_bounds__(WGM * WGN * 64) void gemm_mfma_kernel(GemmParams p) {
  constexpr int WTM = BM / WGM, WTN = BN / WGN;
  constexpr int TM = WTM / 32, TN = WTN / 32;
  constexpr int NWAVES = WGM * WGN;
  constexpr int KS = BK / 16;  // 16-wide k-steps per K step
  constexpr int A_BYTES = BM * BK * 2, B_BYTES = BN * BK * 2;
  constexpr int STAGE = A_BYTES + B_BYTES;
  typedef typename Elem<T>::vec8 V8;
  typedef Loader<A_MC, BM, BK, NWAVES> LoaderA;
  typedef Loader<B_MC, BN, BK, NWAVES> LoaderB;
  __shared__ __attribute__((aligned(1024))) char lds[NSTAGE * STAGE];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;

  request_first_args(p);
  const TileAt tile = tile_at(blockIdx.x, p.order);
  const int m0 = tile.m * BM, n0 = tile.n * BN;

  const int64_t bz = blockIdx.z;
  const int64_t k0 = bz * p.kslice;  // K slices (kslice > 0): grid member z takes k0 .. k0 + kslice - 1
  const int K = p.kslice ? min(p.K - (int)k0, p.kslice) : p.K;
  const T* A = reinterpret_cast<const T*>(p.a) + bz * p.sa + (A_MC ? k0 * p.lda : k0);
  const T* B = reinterpret_cast<const T*>(p.b) + bz * p.sb + (B_MC ? k0 * p.ldb : k0);

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = zero16();

  LoaderA la;
  LoaderB lb;
  const int KT = (K + BK - 1) / BK;
  la.init(p.lda, p.M - m0, wave, lane);
  lb.init(p.ldb, p.N - n0, wave, lane);
  // Tile origins; one K step further is +BK elements (KC) or +BK rows (MC).
  const T* a_tile = A_MC ? A + m0 : A + (int64_t)m0 * p.lda;
  const T* b_tile = B_MC ? B + n0 : B + (int64_t)n0 * p.ldb;
  const int64_t a_step = A_MC ? BK * p.lda : BK;
  const int64_t b_step = B_MC ? BK * p.ldb : BK;
  constexpr int LOADS = LoaderA::NL + LoaderB::NL;  // per wave per K step

  // Prologue: K steps 0 .. NSTAGE-2 go to stages 0 .. NSTAGE-2.  Loads past the end of K are
  // out of range and write zeros, so every step issues the same number of loads and the
  // vmcnt arithmetic below is uniform.
#pragma unroll
  for (int st = 0; st < NSTAGE - 1; ++st) {
    la.issue(a_tile, K - st * BK, lds + st * STAGE, wave);
    lb.issue(b_tile, K - st * BK, lds + st * STAGE + A_BYTES, wave);
    a_tile += a_step;
    b_tile += b_step;
  }
  __builtin_amdgcn_s_waitcnt(vmcnt_imm((NSTAGE - 2) * LOADS));  // step 0 has landed (loads return in order)
  __builtin_amdgcn_s_barrier();

  FragAddr<A_MC, BM, BK, TM> faddr;
  FragAddr<B_MC, BN, BK, TN> fbddr;
  faddr.init(wm * WTM, lane);
  fbddr.init(wn * WTN, lane);

  // Fragments are double-buffered in registers: while the matrix cores work on k-step ks,
  // the LDS reads of k-step ks+1 are in flight.
  V8 fa[2][TM], fb[2][TN];
  auto read_frags = [&](const char* __restrict__ stage, int ks, int buf) {
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[buf][i] = faddr.template read<V8>(stage, i, ks);
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[buf][j] = fbddr.template read<V8>(stage + A_BYTES, j, ks);
  };
  auto mma = [&](int buf) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int jj = (i & 1) ? TN - 1 - j : j;  // boustrophedon: consecutive MFMAs share one operand
        acc[i][jj] = Elem<T>::mfma(fb[buf][jj], fa[buf][i], acc[i][jj]);
      }
  };
  constexpr int READS = (A_MC ? 2 : 1) * TM + (B_MC ? 2 : 1) * TN;
  constexpr int NMFMA = TM * TN;
  // Instruction mix of one k-step: after every MFMA one LDS read (while there are any) and,
  // spread evenly over the MFMAs, `nloads` global loads.
  auto interleave = [&](int nloads) {
#pragma unroll
    for (int r = 0; r < NMFMA; ++r) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                 // 1 MFMA
      if (r < READS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // 1 DS read
      if ((r + 1) * nloads / NMFMA > r * nloads / NMFMA)
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);               // 1 VMEM read
    }
  };
  // One K step: compute from stage `cur`, prefetch the first fragments of stage `nxt`, and fill
  // stage `wr` with K step kt + NSTAGE - 1.  The three stages are distinct; saying so
  // (__restrict__) lets the compiler keep the LDS-DMA loads in flight across the fragment reads
  // instead of waiting for them before every LDS read.  What must be waited for is written out:
  // before the barrier, all but the youngest (NSTAGE-2) steps' loads of this wave have landed
  // (loads return in order), so step kt + 1 is complete once every wave has arrived, and this
  // wave's reads of `cur` are done, so `cur` may be overwritten by the loads the next step issues.
  auto k_step = [&](auto CHECK, const char* __restrict__ cur, const char* __restrict__ nxt, char* __restrict__ wr,
                    int kt) {
    constexpr bool CHECK_K = decltype(CHECK)::value;
    const int kleft = K - (kt + NSTAGE - 1) * BK;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(a_tile), rb = make_rsrc(b_tile);
    static_for<KS>([&](auto KSI) {
      constexpr int ks = decltype(KSI)::value;
      // this k-step's share of the loads
      constexpr int la0 = LoaderA::NL * ks / KS, la1 = LoaderA::NL * (ks + 1) / KS;
      constexpr int lb0 = LoaderB::NL * ks / KS, lb1 = LoaderB::NL * (ks + 1) / KS;
      if constexpr (ks + 1 == KS) {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((NSTAGE - 3) * LOADS + LoaderA::NL * ks / KS + LoaderB::NL * ks / KS) &
                                   ~(0xf << 8));  // and lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
      }
#pragma unroll
      for (int i = la0; i < la1; ++i) la.template issue_one<CHECK_K>(i, ra, kleft, wr, wave);
#pragma unroll
      for (int i = lb0; i < lb1; ++i) lb.template issue_one<CHECK_K>(i, rb, kleft, wr + A_BYTES, wave);
      if constexpr (ks + 1 < KS) read_frags(cur, ks + 1, (ks + 1) & 1);
      else read_frags(nxt, 0, KS & 1);
      mma(ks & 1);
      interleave((la1 - la0) + (lb1 - lb0));
      __builtin_amdgcn_sched_barrier(0);
    });
    a_tile += a_step;
    b_tile += b_step;
  };

  static_assert(KS % 2 == 0, "fragment double-buffering assumes an even number of k-steps");
  static_assert(NSTAGE >= 3, "the barrier leaves the running step's loads in flight");
  read_frags(lds, 0, 0);
  // Step kt loads K step kt + NSTAGE - 1: all of it exists until that index reaches the last
  // (possibly partial) step, so only the final NSTAGE - 1 iterations (and a partial last K step)
  // need the per-lane K test.
  const int kt_full = min(KT, K / BK - (NSTAGE - 1));
  int kt = 0;
  if constexpr (NSTAGE == 4) {
    for (; kt < kt_full; ++kt)
      k_step(std::false_type{}, lds + (kt % NSTAGE) * STAGE, lds + ((kt + 1) % NSTAGE) * STAGE,
             lds + ((kt + NSTAGE - 1) % NSTAGE) * STAGE, kt);
    for (; kt < KT; ++kt)
      k_step(std::true_type{}, lds + (kt % NSTAGE) * STAGE, lds + ((kt + 1) % NSTAGE) * STAGE,
             lds + ((kt + NSTAGE - 1) % NSTAGE) * STAGE, kt);
  } else {
    // The stages' offsets are carried along: kt % 3 is a chain of scalar multiplications in front of every step's LDS
    // addresses (256 x 128 tile: 2048 x 4096 x 4096 61.0 -> 58.4 us; with four stages it is a mask, and the faster form).
    int cur = 0, nxt = STAGE, wr = (NSTAGE - 1) * STAGE;
    auto turn = [&] {
      wr = cur;
      cur = nxt;
      nxt = nxt == (NSTAGE - 1) * STAGE ? 0 : nxt + STAGE;
    };
    for (; kt < kt_full; ++kt, turn()) k_step(std::false_type{}, lds + cur, lds + nxt, lds + wr, kt);
    for (; kt < KT; ++kt, turn()) k_step(std::true_type{}, lds + cur, lds + nxt, lds + wr, kt);
  }
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // drain the zero-fill loads before LDS is released

  // Epilogue.  acc[i][j][e] is out[m][n] with m = m0 + wm WTM + 32 i + lane%32 and
  // n = n0 + wn WTN + 32 j + 8 (e/4) + 4 (lane/32) + e%4.
  static_assert(NSTAGE * STAGE >= NWAVES * TN * 4096, "a slab per wave is staged in the operand stages");
  __builtin_amdgcn_s_barrier();  // every wave has read its last fragments
  GemmEpilogue<T, OutF32> epi(p, bz);
  store_tile<T, OutF32>(epi, acc, lds + wave * (TN * 4096), member_out(p, bz), p.ldc, bz * p.sc, p.M, p.N, m0 + wm * WTM, n0 + wn * WTN,
                        lane);
}

// Tile policies, the counterpart of the reference's gemm_policy list
// (xetla/gemm/gemm_dispatch.h:183-214).
struct Policy {
  const char* name;
  int bm, bn, wgm, wgn, bk, stages;
  bool alone;          // one work-group fills a CU (LDS)
  bool any_alignment;  // also a tile of the kernels that take any alignment (gemm_ragged.h, gemm_slices.h)
};
constexpr Policy kPolicies[] = {
    {"mfma_256x256x32_w2x2_s4", 256, 256, 2, 2, 32, 4, true, false},
    // (four stages of the 128 x 128 tile against three: 512 x 4096 x 4096 with B [n,k] 28.6 -> 24.8 us, 4096^3 135.8 -> 129.0)
    {"mfma_128x128x64_w2x2_s4", 128, 128, 2, 2, 64, 4, true, true},
    {"mfma_128x64x64_w2x2_s4", 128, 64, 2, 2, 64, 4, true, false},
    {"mfma_64x64x64_w2x2_s4", 64, 64, 2, 2, 64, 4, false, true},
    {"mfma_256x128x64_w2x2_s3", 256, 128, 2, 2, 64, 3, true, false},
    // not a matrix-core tile: the streaming kernel for up to eight rows (gemm_rows.hip), eight waves
    // that split the reduction of a 512-column block
    {"stream_rows_8x512_w8", 8, 512, 8, 1, 8, 2, true, false},
    // small tiles whose reduction is split over the waves of a work-group (gemm_slices.h)
    {"slices_32x32_w4", 32, 32, 4, 1, 64, 2, false, true},
    {"slices_32x32_w8", 32, 32, 8, 1, 64, 2, true, true},
    {"slices_32x32_w16", 32, 32, 16, 1, 64, 2, true, true},
    {"slices_32x64_w8", 32, 64, 8, 1, 64, 2, true, true},
    {"slices_64x64_w4", 64, 64, 4, 1, 64, 2, false, true},
    {"slices_64x64_w8", 64, 64, 8, 1, 64, 2, true, true},
    // between the 128 x 128 and the 256 x 128 tile, for outputs that those leave CUs idle or nearly empty rounds with:
    // 1152 x 4096 x 4096 47.8 -> 40.7 us, 768 x 8192 x 4096 (B [n,k]) 60.6 -> 52.6, 1024 x 5056 x 2048 28.9 -> 26.7
    {"mfma_192x128x64_w2x2_s4", 192, 128, 2, 2, 64, 4, true, false},
    // three work-groups on a CU, so that one's epilogue runs beside the others' loads and products: large outputs of short
    // reductions, where a tile alone on its CU does one after the other (8072 x 4544 x 256 50.8 -> 33.1 us, 7553 x 2640 x 152
    // 31.5 -> 19.7, 3094 x 6104 x 504 46.4 -> 35.9; 4096^3 150.8 against 110).  256 x 128 likewise, two of them: ahead of all
    // others by 6 % on one shape in fifty, left out.
    {"mfma_128x128x32_w2x2_s3", 128, 128, 2, 2, 32, 3, false, false},
};
constexpr int kNumPolicies = sizeof(kPolicies) / sizeof(kPolicies[0]);
constexpr int kRowsPolicy = 5;
constexpr int kSlicesPolicy = 6;        // first of the slices variants
constexpr int kNumSlices = 6;
constexpr bool is_slices(int policy) { return policy >= kSlicesPolicy && policy < kSlicesPolicy + kNumSlices; }
constexpr int k192Policy = 12, k3PerCuPolicy = 13;
constexpr int kRowsMaxM = 8;            // rows the streaming kernel takes
constexpr int kRowsMinBN = 64;          // its output columns per work-group: 64, 128, 256 or 512
constexpr int kRowsEnoughBlocks = 192;  // work-groups from which on a launch pulls the memory system's rate
// The streaming kernel is the default where 128-column blocks are already that many work-groups, i.e. from
// 24.5 thousand columns on (the vocabulary projections).  Measured, fp16, k = 4096, microseconds, best
// matrix-core choice against best streaming choice: n = 50400, m = 4: 96.9 / 71.9 (5.75 TB/s); n = 16384,
// m = 1: 27.7 / 28.5, m = 4: 27.4 / 31.1; n = 12288, m = 8: 25.9 / 32.2; n = 4096, k = 16384, m = 4:
// 30.1 / 36.8: below that width a launch is over before the stream has paid for its start and end.
constexpr int kRowsDefaultBN = 128;
// B stored [N, K] streams in blocks of 64 output columns and is the default for up to four rows from 12288
// columns on (fp16, k = 4096, microseconds, matrix-core kernel against streaming: n = 50400, m = 1: 89.2 /
// 78.6, m = 4: 90.1 / 80.8, m = 8: 91.4 / 95.6; n = 32000, m = 4: 61.6 / 49.5; n = 16384, m = 4: 33.6 / 25.5).
constexpr int kColsBN = 64;
constexpr int kColsMaxK = 16384;  // reduction length its register-resident pieces of A allow
enum : int { kRowsNone = 0, kRowsMC = 1, kRowsKC = 2 };  // which streaming kernel the operands allow

// Tile choice, the role of selectXetlaGemmConfig (xetla/gemm/gemm.cc:286-308).  Shapes listed in the tuned table
// (gemm_policy_table.h, written by autotune_gemm.py from measurements) take the policy
// recorded there, as the reference's configMap does (gemm.cc:31-285).
// XMK_GEMM_POLICY forces one policy for every shape (what the autotuner uses).
// ksplit: K slices to use when the caller supplies scratch (xmk_gemm_ws); 0 = no tuned value, the
// planner's own rule decides.  With ksplit > 1 `policy` is the tile of the slices.
struct TunedShape {
  int m, n, k, policy, ksplit;
};
#include "gemm_policy_table.h"
inline const TunedShape* tuned_shape(int64_t m, int64_t n, int64_t k) {
  for (const TunedShape& t : kTunedShapes)
    if (t.m == m && t.n == n && t.k == k) return &t;
  return nullptr;
}
inline bool rows_streams_by_default(int rows_kind, int64_t m, int64_t n) {
  return (rows_kind == kRowsMC && xmk::ceil_div(n, (int64_t)kRowsDefaultBN) >= kRowsEnoughBlocks) ||
         (rows_kind == kRowsKC && m <= 4 && xmk::ceil_div(n, (int64_t)kColsBN) >= kRowsEnoughBlocks);
}
// XMK_GEMM_POLICY=<index>; kByRule where it is negative (the choice without the tuned table, which the autotuner compares
// with); kUnforced where it is not set.  Read at every call (a getenv costs far less than a launch), so that the autotuner
// can walk the policies inside one process.
enum : int { kUnforced = -1, kByRule = -2 };
inline int forced_policy() {
  const char* e = getenv("XMK_GEMM_POLICY");
  if (!e || !*e) return kUnforced;
  const int v = atoi(e);
  return v < 0 ? kByRule : v < kNumPolicies ? v : kUnforced;
}
// Which kernels a product's operands allow, and which cost table below applies.
enum : int { kClassKN = 0, kClassNK = 1, kClassRagged = 2, kClassF32 = 3 };

// Estimated microseconds of a launch: with KT K steps of 128 bytes, KTw = ceil(KT / waves that split K) of them per
// wave, and L output tiles per CU (the mean of the tiles / 256 and, for kernels of which one work-group fills a CU,
// that rounded up; at least 1),
//     start + step * KTw + fill * KT * min(tiles / 256, 1) / 8 + (L - 1) * (more_step * KT + more).
// Least-squares fits (non-negative, relative error) to 380 shapes per class, m 1 .. 8192, n and k 64 .. 16384 at
// random, every policy: mean error 5 - 12 %.  They are older than the fourth stage of the 128 x 128 tile and the present tile
// order.  With these, on 1100 to 1250 other shapes per class, the weights from memory, the policy that this picks is without a
// K split 3.2 % slower than the best of all ([k,n]; [n,k] 3.1 %, any alignment 1.7 %, fp32 1.9 %), one in ten by more than 5 to
// 7 %, the worst by 78 % (609 x 1568 x 6968; the streaming kernel for [n,k] apart: 4 x 13536 x 80 takes it 14 us, a tile 4).
// With scratch, against every tile on 1 to 8 slices, 500 to 730 shapes per class, it is level on aligned operands (copies and
// streams are no tiles), any alignment and fp32 3 %, one in ten by more than 7 to 10 %, the worst by 34 %.
// The last two tiles' rows: chosen for what they pick beside the others.  192 x 128, on 855 shapes of more than 100 tiles of
// 128 x 128: taken for 200 of them, 13 % faster there on average, nine 2 to 5 % slower.  128 x 128 in steps of 32, on 900 of
// more than 40, k 64 .. 8192: taken for 180, 30 % faster there.  Both on 1520 others of more than 200 and k 64 .. 3000, either
// storage order of both operands, against the choice without the two: 10 % faster on average, eight of the 1520 more than 3 %
// slower (1656 x 4760 x 552 with B [n,k] 12 %, the others 6 % and less).
// Looking all candidates over takes the host 0.15 to 0.65 us per call.
struct TileCost {
  float start, step, more_step, more, fill;
};
constexpr TileCost kTileCost[4][kNumPolicies] = {
    {  // 16-bit direct, B stored [K, N]
     {8.351f, 0.951f, 1.639f, 13.748f, 4.611f},
     {4.75f, 0.383f, 0.581f, 4.353f, 1.658f},
     {3.917f, 0.227f, 0.359f, 2.594f, 1.268f},
     {3.311f, 0.176f, 0.264f, 0.864f, 1.132f},
     {6.284f, 0.544f, 0.927f, 7.589f, 2.347f},
     {},
     {3.046f, 0.4f, 0.134f, 0.51f, 0.997f},
     {2.739f, 0.775f, 0.133f, 0.904f, 1.128f},
     {2.414f, 1.588f, 0.142f, 2.431f, 1.071f},
     {2.953f, 1.099f, 0.213f, 2.398f, 1.076f},
     {3.747f, 0.862f, 0.313f, 3.855f, 1.603f},
     {3.11f, 1.488f, 0.285f, 3.156f, 1.679f},
     {4.669f, 0.509f, 0.831f, 4.313f, 1.555f},
     {3.941f, 0.676f, 0.578f, 0.601f, 1.348f},
    },
    {  // 16-bit direct, B stored [N, K]
     {8.272f, 0.959f, 1.836f, 11.842f, 5.729f},
     {4.462f, 0.33f, 0.572f, 4.093f, 2.144f},
     {3.935f, 0.233f, 0.359f, 2.565f, 1.197f},
     {3.294f, 0.181f, 0.264f, 0.822f, 1.065f},
     {6.1f, 0.504f, 0.92f, 7.263f, 2.622f},
     {},
     {3.126f, 0.344f, 0.115f, 0.396f, 0.677f},
     {2.961f, 0.618f, 0.116f, 0.923f, 0.773f},
     {2.642f, 1.273f, 0.127f, 2.333f, 0.754f},
     {2.982f, 1.019f, 0.208f, 2.326f, 1.129f},
     {3.735f, 0.806f, 0.31f, 3.754f, 1.666f},
     {2.945f, 1.596f, 0.302f, 3.078f, 2.018f},
     {4.41f, 0.482f, 0.815f, 3.821f, 1.96f},
     {4.065f, 0.485f, 0.6f, 1.552f, 3.272f},
    },
    {  // 16-bit, any alignment
     {},
     {5.669f, 0.788f, 0.716f, 2.853f, 1.6f},
     {},
     {3.676f, 0.372f, 0.345f, 0.464f, 1.275f},
     {},
     {},
     {3.458f, 0.555f, 0.191f, 0.405f, 0.898f},
     {3.075f, 1.115f, 0.217f, 1.339f, 1.047f},
     {2.134f, 2.386f, 0.219f, 2.215f, 0.885f},
     {3.127f, 1.701f, 0.27f, 2.754f, 1.078f},
     {4.579f, 1.086f, 0.361f, 4.139f, 1.668f},
     {3.475f, 2.21f, 0.388f, 3.206f, 1.537f},
    },
    {  // fp32
     {},
     {6.542f, 0.829f, 1.369f, 8.845f, 5.211f},  // fitted again, to 70 shapes of 24 tiles and more (6 % mean error)
     {},
     {3.391f, 0.597f, 0.512f, 1.128f, 0.934f},
     {},
     {},
     {3.307f, 0.657f, 0.155f, 0.72f, 0.466f},
     {3.068f, 1.181f, 0.16f, 1.243f, 0.639f},
     {2.366f, 2.376f, 0.17f, 2.807f, 0.659f},
     {3.185f, 2.181f, 0.291f, 3.548f, 0.841f},
     {4.218f, 2.231f, 0.586f, 5.833f, 1.448f},
     {2.873f, 4.47f, 0.562f, 5.601f, 1.5f},
    },
};
// What a K split adds for its second launch, and the least it takes end to end when launched from a host program.
constexpr float kSplitCost = 4.0f, kSplitFloor = 8.0f;

// kt: K steps of 128 bytes.
inline float launch_cost(const Policy& P, const TileCost& c, bool slices, uint32_t m, uint32_t n, uint32_t kt, uint32_t batch) {
  auto blocks = [](uint32_t v, int b) {  // b: a power of two, or three times one
    const int shift = __builtin_ctz((unsigned)b);
    const uint32_t units = (v + (1u << shift) - 1) >> shift;
    return b >> shift == 3 ? (units + 2) / 3 : units;
  };
  const uint64_t tiles = (uint64_t)blocks(m, P.bm) * blocks(n, P.bn) * batch;
  const float load = (float)tiles * (1.0f / 256);
  const uint32_t ktw = slices ? blocks(kt, P.wgm) : kt;
  const float l = P.alone ? 0.5f * (load + (float)((tiles + 255) >> 8)) : load;
  return c.start + c.step * (float)ktw + c.fill * (float)kt * (load < 1.0f ? load : 1.0f) * 0.125f +
         (l > 1.0f ? l - 1.0f : 0.0f) * (c.more_step * (float)kt + c.more);
}

struct Choice {
  int policy, slices;
  float us;
};
// The cheapest policy and number of K slices (1 unless may_split).  a_mc: A is stored [K, M].
inline Choice cheapest(int64_t m, int64_t n, int64_t k, int64_t batch, int cls, bool may_split, bool a_mc = false) {
  Choice best{3, 1, 1e30f};
  const bool direct = cls == kClassKN || cls == kClassNK;
  const int kstep = cls == kClassF32 ? 32 : 64;
  const int64_t tiles_256_x_256 = xmk::ceil_div(m, 256) * xmk::ceil_div(n, 256) * batch;
  const int64_t tiles_192_x_128 = xmk::ceil_div(m, 192) * xmk::ceil_div(n, 128) * batch;
  auto each = [&](int s, float extra, float least) {
    for (int pol = 0; pol < kNumPolicies; ++pol) {
      if (pol == kRowsPolicy || (!direct && !kPolicies[pol].any_alignment) || (a_mc && pol == k192Policy)) continue;
      const uint32_t kt = (uint32_t)(((k + s - 1) / s + kstep - 1) / kstep);
      // The 192 x 128 tile is not for short reductions, whose time is the output's (7102 x 1408 x 64 11 % slower), nor for long ones
      // where the 256-row tile takes as many: the last of that one's tile rows is the emptier, which gives the others clock and
      // load path (560 x 10240 x 12288 141 us against 159; 560 x 10240 x 2048 30.1 against 27.3).
      // With K slices its estimate is too low (161 x 3553 x 12725 62.8 us, with it 72.4).
      // 128 x 128 in steps of 32: not with K slices, of which it is the slowest tile (1024 x 1024 x 8192 on four 39.0 us, in steps
      // of 64 30.3; 2048 x 2048 x 4096 on two 61 and 64, unsplit 35).
      // Nor, above six K steps, where the 256 x 256 tiles are more than a round and a half: they load half as much, and the estimate
      // did not see it (5400 x 15512 x 840 202 us where they take 168, 6936 x 8152 x 560 with B [n,k] 109 against 93).
      if (pol == k3PerCuPolicy && (s > 1 || (kt > 6 && tiles_256_x_256 > 384))) continue;
      if (pol == k192Policy && (s > 1 || kt < 6 || (kt > 32 && xmk::ceil_div(m, 192) == xmk::ceil_div(m, 256)))) continue;
      float us = launch_cost(kPolicies[pol], kTileCost[cls][pol], is_slices(pol), (uint32_t)m, (uint32_t)n, kt, (uint32_t)(batch * s));
      // A second round of fewer than a hundred 192 x 128 tiles takes longer than the estimate's share of one: 5 % on it gives such
      // sizes to others (568 x 11568 x 1112 33.6 -> 24.2 us, 528 x 12400 x 1328 36.3 -> 27; over 700 sizes of 257 to 384 of the
      // tiles 0.4 % on the mean, and the worst loss against having no such tile 12 % where it was 39).
      if (pol == k192Policy && tiles_192_x_128 > 256 && tiles_192_x_128 <= 352) us *= 1.05f;
      const float cost = std::max(us + extra, least);
      if (cost < best.us) best = {pol, s, cost};
    }
  };
  each(1, 0.0f, 0.0f);
  for (int s = 2; may_split && s <= 16 && best.us > kSplitFloor; s *= 2) {
    if (k / s < 128 || (float)m * (float)n * (float)s > 6.4e7f) break;
    each(s, kSplitCost + (float)m * (float)n * (float)s * (8.0f / 3e6f), kSplitFloor);
  }
  return best;
}

// rows_kind: which streaming kernel the operands allow (gemm_rows_applicable); it is never chosen otherwise.
// The tuned table applies to the layout it was measured with (direct operands, B stored [K, N]).
inline int select_policy(int64_t m, int64_t n, int64_t k, int64_t batch, int rows_kind, int cls, bool a_mc) {
  const bool rows_ok = rows_kind != kRowsNone;
  const bool direct = cls == kClassKN || cls == kClassNK;
  auto usable = [&](int v) {
    return v >= 0 && v < kNumPolicies && (v != kRowsPolicy || rows_ok) && (direct || kPolicies[v].any_alignment) && !(a_mc && v == k192Policy);
  };
  const int forced = forced_policy();
  if (usable(forced)) return forced;
  if (batch == 1 && cls == kClassKN && forced != kByRule)
    if (const TunedShape* t = tuned_shape(m, n, k); t && t->ksplit <= 1 && usable(t->policy)) return t->policy;
  // A few rows against a very wide matrix: stream it.
  if (batch == 1 && rows_streams_by_default(rows_kind, m, n)) return kRowsPolicy;
  return cheapest(m, n, k, batch, cls, false, a_mc).policy;
}

template <typename T, bool OutF32, bool A_MC, bool B_MC, int BM, int BN, int WGM, int WGN, int BK, int NSTAGE>
void launch_mfma(const GemmParams& p, int batch, hipStream_t st) {
  hipLaunchKernelGGL((gemm_mfma_kernel<T, OutF32, A_MC, B_MC, BM, BN, WGM, WGN, BK, NSTAGE>),
                     dim3(p.tiles_m * p.tiles_n, 1, batch), dim3(WGM * WGN * 64), 0, st, p);
}

template <typename T, bool OutF32, bool A_MC, bool B_MC>
void launch_policy(int pol, GemmParams& p, int batch, hipStream_t st) {
  p.tiles_m = (int)xmk::ceil_div(p.M, kPolicies[pol].bm);
  p.tiles_n = (int)xmk::ceil_div(p.N, kPolicies[pol].bn);
  p.order = tile_order((uint32_t)p.tiles_m, (uint32_t)p.tiles_n, p.K);
  switch (pol) {
    case 0: launch_mfma<T, OutF32, A_MC, B_MC, 256, 256, 2, 2, 32, 4>(p, batch, st); break;
    case 1: launch_mfma<T, OutF32, A_MC, B_MC, 128, 128, 2, 2, 64, 4>(p, batch, st); break;
    case 2: launch_mfma<T, OutF32, A_MC, B_MC, 128, 64, 2, 2, 64, 4>(p, batch, st); break;
    case 4: launch_mfma<T, OutF32, A_MC, B_MC, 256, 128, 2, 2, 64, 3>(p, batch, st); break;
    case k3PerCuPolicy: launch_mfma<T, OutF32, A_MC, B_MC, 128, 128, 2, 2, 32, 3>(p, batch, st); break;
    case k192Policy:  // (not for A stored [K, M], whose LDS rows of 192 elements are no whole number of loads)
      if constexpr (!A_MC) launch_mfma<T, OutF32, A_MC, B_MC, 192, 128, 2, 2, 64, 4>(p, batch, st);
      break;
    default: launch_mfma<T, OutF32, A_MC, B_MC, 64, 64, 2, 2, 64, 4>(p, batch, st); break;
  }
}

template <typename T, bool OutF32>
void launch_layout_impl(bool a_mc, bool b_mc, int pol, GemmParams& p, int batch, hipStream_t st) {
  if (!a_mc && !b_mc) launch_policy<T, OutF32, false, false>(pol, p, batch, st);
  else if (!a_mc && b_mc) launch_policy<T, OutF32, false, true>(pol, p, batch, st);
  else if (a_mc && !b_mc) launch_policy<T, OutF32, true, false>(pol, p, batch, st);
  else launch_policy<T, OutF32, true, true>(pol, p, batch, st);
}

// Explicitly instantiated in gemm_inst_*.hip.
template <typename T, bool OutF32>
void launch_layout(bool a_mc, bool b_mc, int pol, GemmParams& p, int batch, hipStream_t st);

}  // namespace gemm_impl
