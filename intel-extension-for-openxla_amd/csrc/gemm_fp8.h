// fp8 (OCP e4m3fn) element type of the kernels that take any alignment, and what fp8_gemm.hip shares with them.
#pragma once
#include "gemm_ragged.h"
#include "gemm_slices.h"

namespace gemm_impl {

struct Fp8 { uint8_t bits; };
typedef int intx8 __attribute__((ext_vector_type(8)));

// bias (bf16 [N]) and c come with GemmParams; c is not used.
struct Fp8Params : GemmParams {
  const float* a_scale;
  const float* b_scale;
  const float* d_scale;  // optional: multiplies the result after the bias
};

__device__ __forceinline__ floatx16 mfma_fp8(intx8 a, intx8 b, floatx16 c) {
  // cbsz = blgp = 0: both operands e4m3; block scales 127 = 2^0 (E8M0).
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 127, 0, 127);
}

// out element = bf16(d_scale * (a_scale * b_scale * acc + bias[n])); `scale` = a_scale * b_scale.
struct Fp8Epilogue {
  float scale, post;
  const __bf16* bias;
  float b[8];  // the bias of the lane's columns (store_tile)
  __device__ __forceinline__ explicit Fp8Epilogue(const Fp8Params& p, int64_t = 0)
      : scale(p.a_scale[0] * p.b_scale[0]), post(p.d_scale ? p.d_scale[0] : 1.0f), bias(reinterpret_cast<const __bf16*>(p.bias)) {}
  __device__ __forceinline__ __bf16 operator()(float acc, int n) const {
    float v = acc * scale;
    if (bias) v += (float)bias[n];
    return (__bf16)(v * post);
  }
  __device__ __forceinline__ void columns(int n, int count) {
    if (bias && count > 0) GemmEpilogue<__bf16, false>::fetch<false>(bias, n, count, b);
  }
  template <int U>
  __device__ __forceinline__ void apply(float (&v)[U][8], const int (&)[U], int, int) const {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        v[u][e] *= scale;
        if (bias) v[u][e] += b[e];
        v[u][e] *= post;
      }
  }
};

template <> struct Elem<Fp8> {
  typedef intx8 vec8;  // 32 consecutive k
  static __device__ __forceinline__ floatx16 mfma(intx8 a, intx8 b, floatx16 c) { return mfma_fp8(a, b, c); }
};
template <> struct AnyType<Fp8> {
  typedef Fp8Params Params;
  typedef __bf16 Out;
  static constexpr int KS = 2;
  template <bool OutF32> using Epilogue = Fp8Epilogue;
};

// Half ks of a K step: lane l holds row l % 32, k = 64 ks + 32 (l / 32) .. +31.
//   KC: two neighbouring 16-byte chunks.
//   MC: four transpose reads, 8 rows of k apart; within a block of 16 lanes, lane p addresses row kb + p / 2, bytes
//       cb + 8 (p % 2) .. +7 and receives column cb + p, rows kb .. kb + 7.
template <bool MC, int ROWS, int TT>
struct AnyFrag<Fp8, MC, ROWS, TT> {
  typedef intx8 V;
  int base[MC ? TT * 4 : 4];
  __device__ __forceinline__ void init(int row0, int lane) {
    if constexpr (MC) {
      const int p = lane & 15;
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int k = (lane >> 5) * 32 + 8 * q + (p >> 1);  // + 64 ks, which does not change the swizzle
          const int col = row0 + t * 32 + ((lane >> 4) & 1) * 16 + 8 * (p & 1);
          base[t * 4 + q] = k * ROWS + (((col >> 4) ^ AnyLoader<Fp8, true, ROWS, 64, true>::swizzle(k)) << 4) + (col & 15);
        }
    } else {
      const int row = row0 + (lane & 31);
#pragma unroll
      for (int c = 0; c < 4; ++c) base[c] = row * 128 + (((4 * (c >> 1) + 2 * (lane >> 5) + (c & 1)) ^ swz<false, ROWS, 64>(row)) << 4);
    }
  }
  __device__ __forceinline__ V read(const char* tile, int t, int ks) const {
    V v;
    if constexpr (MC) {
      typedef int int2v __attribute__((ext_vector_type(2)));
      typedef int2v __attribute__((address_space(3))) * lds_ptr;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int2v r = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_ptr)(tile + base[t * 4 + q] + ks * 64 * ROWS));
        v[2 * q] = r[0];
        v[2 * q + 1] = r[1];
      }
    } else {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const u32x4 w = *reinterpret_cast<const u32x4*>(tile + base[2 * ks + c] + t * 4096);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * c + e] = (int)w[e];
      }
    }
    return v;
  }
};

// The fp8 product's tiles.  0 .. 2: the direct-to-LDS kernel of fp8_gemm.hip; the others take any alignment.
// ("alone" where the estimates fit better so, also of tiles of which two share a CU.)
constexpr Policy kFp8Policies[] = {
    {"mfma_256x256", 256, 256, 2, 4, 64, 4, true, false},
    {"mfma_256x128", 256, 128, 2, 2, 64, 4, true, false},
    {"mfma_128x128", 128, 128, 2, 2, 64, 4, true, false},
    {"any_128x128", 128, 128, 2, 2, 128, 2, true, true},
    {"any_64x64", 64, 64, 2, 2, 128, 2, false, true},
    {"slices_32x32_w4", 32, 32, 4, 1, 128, 2, true, true},
    {"slices_32x32_w8", 32, 32, 8, 1, 128, 2, true, true},
    {"slices_32x32_w16", 32, 32, 16, 1, 128, 2, true, true},
    {"slices_32x64_w8", 32, 64, 8, 1, 128, 2, true, true},
    {"slices_64x64_w4", 64, 64, 4, 1, 128, 2, true, true},
    {"slices_64x64_w8", 64, 64, 8, 1, 128, 2, true, true},
};
constexpr int kFp8Policies_n = sizeof(kFp8Policies) / sizeof(kFp8Policies[0]);
constexpr int kFp8Direct = 3, kFp8Slices = 5;

// Estimated microseconds (launch_cost in gemm_kernel.h), fitted to 6100 shapes per direct class and 3200 of the other, m 1 .. 8192,
// n 64 .. 16384, k 64 .. 16384, weights from memory: least squares, then moved so that the policies they choose are the fastest.
// On 1500 (800) other shapes 0.6 % (0.5 %) from the best policy of all measured, one in ten more than 2 %, the worst 21 % (24 %).
// A table fitted to k of 256 and more, which stood here before, lost 4 to 5 % (3 %), one in ten 12 to 14 % (8 %): 965 x 5456 x 96, B
// [k,n], 10.4 us on 128 x 128 tiles where 64 x 64 take 7.8.
constexpr TileCost kFp8Cost[3][kFp8Policies_n] = {
    {  // direct loads possible, B stored [K, N]
     {7.4f, 0.974f, 1.068f, 9.869f, 8.691f},
     {5.27f, 0.759f, 0.835f, 6.426f, 11.51f},
     {3.83f, 0.888f, 0.745f, 1.616f, 0.024f},  // (more than 256 tiles)
     {4.299f, 0.695f, 0.488f, 2.753f, 1.793f},
     {3.311f, 0.326f, 0.3f, 0.355f, 1.468f},
     {2.551f, 0.469f, 0.163f, 0.129f, 1.093f},
     {1.394f, 1.516f, 0.262f, 1.148f, 1.31f},
     {0.307f, 4.123f, 0.241f, 1.936f, 2.128f},
     {2.035f, 1.596f, 0.203f, 2.081f, 1.276f},
     {3.352f, 1.037f, 0.361f, 3.278f, 1.494f},
     {2.437f, 2.515f, 0.399f, 3.198f, 3.169f},
    },
    {  // direct loads possible, B stored [N, K]
     {7.227f, 0.979f, 1.902f, 9.457f, 9.902f},
     {4.898f, 0.721f, 0.874f, 6.179f, 12.309f},
     {3.75f, 0.975f, 0.746f, 1.457f, 0.067f},  // (more than 256 tiles)
     {4.05f, 0.743f, 0.512f, 2.339f, 2.12f},
     {3.03f, 0.346f, 0.3f, 0.434f, 1.062f},
     {2.024f, 0.448f, 0.12f, 0.326f, 0.694f},
     {2.501f, 0.816f, 0.16f, 1.159f, 0.756f},
     {1.468f, 2.761f, 0.182f, 1.976f, 1.487f},
     {2.671f, 0.858f, 0.188f, 2.071f, 1.393f},
     {3.682f, 0.829f, 0.286f, 3.477f, 1.247f},
     {2.793f, 1.62f, 0.256f, 3.124f, 2.311f},
    },
    {  // any alignment
     {},
     {},
     {},
     {5.682f, 0.818f, 0.484f, 2.523f, 3.206f},
     {3.202f, 0.464f, 0.36f, 0.586f, 1.811f},
     {1.951f, 0.684f, 0.226f, 0.394f, 0.95f},
     {2.952f, 1.299f, 0.315f, 1.144f, 1.562f},
     {1.195f, 3.618f, 0.264f, 3.012f, 2.195f},
     {2.128f, 1.501f, 0.318f, 2.545f, 1.62f},
     {3.91f, 1.244f, 0.47f, 3.883f, 1.945f},
     {3.065f, 3.612f, 0.521f, 4.207f, 2.525f},
    },
};

// The 128 x 128 tile where every CU has one at most (K steps of 128 bytes), B stored [K, N] / [N, K]; fitted with them.
constexpr TileCost kFp8OnePerCu[2] = {{4.287f, 0.509f, 0.016f, 0.f, 2.896f}, {4.124f, 0.487f, 0.055f, 0.f, 3.529f}};

// Policies 3 and up; A is [M, K], b_mc: B stored [K, N].
void launch_fp8_any(int policy, bool b_mc, Fp8Params& p, hipStream_t st);

}  // namespace gemm_impl
