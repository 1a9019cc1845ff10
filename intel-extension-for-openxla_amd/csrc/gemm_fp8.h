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
constexpr Policy kFp8Policies[] = {
    {"mfma_256x256", 256, 256, 2, 4, 64, 4, true, false},
    {"mfma_256x128", 256, 128, 2, 2, 64, 4, true, false},
    {"mfma_128x128", 128, 128, 2, 2, 64, 4, false, false},
    {"any_128x128", 128, 128, 2, 2, 128, 2, false, true},
    {"any_64x64", 64, 64, 2, 2, 128, 2, false, true},
    {"slices_32x32_w4", 32, 32, 4, 1, 128, 2, false, true},
    {"slices_32x32_w8", 32, 32, 8, 1, 128, 2, true, true},
    {"slices_32x32_w16", 32, 32, 16, 1, 128, 2, true, true},
    {"slices_32x64_w8", 32, 64, 8, 1, 128, 2, true, true},
    {"slices_64x64_w4", 64, 64, 4, 1, 128, 2, false, true},
    {"slices_64x64_w8", 64, 64, 8, 1, 128, 2, true, true},
};
constexpr int kFp8Policies_n = sizeof(kFp8Policies) / sizeof(kFp8Policies[0]);
constexpr int kFp8Direct = 3, kFp8Slices = 5;

// Estimated microseconds (launch_cost in gemm_kernel.h).  The direct classes are fitted to 350 shapes each, m 2 .. 8192, n 64 ..
// 16384, k 256 .. 16384, weights from memory: on 115 others per class 3 % from the best policy of all measured, one in ten
// more than 10 %, the worst 34 % (the table before the tiles' present order: [k,n] 7 %, 23 %, 64 %).  The any-alignment class:
// 240 shapes, m 1 .. 8192, 2 % on those, 3 to 4 % on others.
constexpr TileCost kFp8Cost[3][kFp8Policies_n] = {
    {  // direct loads possible, B stored [K, N]
     {5.397f, 0.987f, 1.885f, 8.612f, 5.243f},
     {4.759f, 0.596f, 1.095f, 6.471f, 3.21f},
     {5.059f, 0.806f, 0.561f, 1.5f, 0.f},  // (more than 256 tiles)
     {4.011f, 0.668f, 0.532f, 2.909f, 1.888f},
     {3.027f, 0.32f, 0.225f, 0.672f, 1.311f},
     {3.021f, 0.388f, 0.18f, 0.286f, 1.294f},
     {2.704f, 0.875f, 0.194f, 0.936f, 1.195f},
     {1.231f, 2.745f, 0.246f, 1.699f, 1.428f},
     {2.836f, 1.194f, 0.219f, 1.978f, 1.25f},
     {3.775f, 0.84f, 0.303f, 3.027f, 1.032f},
     {3.356f, 1.986f, 0.388f, 3.034f, 2.102f},
    },
    {  // direct loads possible, B stored [N, K]
     {5.026f, 0.989f, 1.517f, 9.792f, 7.747f},
     {4.458f, 0.597f, 1.115f, 4.438f, 5.174f},
     {4.782f, 0.947f, 0.545f, 1.329f, 0.f},
     {3.78f, 0.644f, 0.521f, 2.042f, 2.495f},
     {3.042f, 0.276f, 0.186f, 0.633f, 1.407f},
     {3.188f, 0.302f, 0.097f, 0.445f, 0.511f},
     {3.186f, 0.579f, 0.122f, 1.073f, 0.565f},
     {2.224f, 1.9f, 0.159f, 1.916f, 0.857f},
     {3.155f, 0.942f, 0.179f, 2.022f, 1.003f},
     {3.749f, 0.766f, 0.282f, 2.87f, 0.995f},
     {3.497f, 1.359f, 0.296f, 2.632f, 1.294f},
    },
    {  // any alignment
     {},
     {},
     {},
     {5.016f, 0.937f, 0.804f, 2.238f, 2.798f},
     {3.469f, 0.413f, 0.383f, 0.587f, 1.429f},
     {2.968f, 0.748f, 0.209f, 0.508f, 0.654f},
     {2.344f, 1.551f, 0.231f, 1.4f, 0.511f},
     {1.357f, 3.735f, 0.293f, 2.856f, 1.51f},
     {2.231f, 2.238f, 0.341f, 2.558f, 0.921f},
     {3.817f, 1.428f, 0.471f, 3.425f, 0.838f},
     {3.23f, 3.795f, 0.64f, 3.87f, 1.223f},
    },
};

// The 128 x 128 tile where every CU has one at most (K steps of 128 bytes), B stored [K, N] / [N, K]; fitted with them.
constexpr TileCost kFp8OnePerCu[2] = {{3.919f, 0.324f, 0.f, 0.f, 2.146f}, {3.689f, 0.29f, 0.f, 0.f, 3.007f}};

// Policies 3 and up; A is [M, K], b_mc: B stored [K, N].
void launch_fp8_any(int policy, bool b_mc, Fp8Params& p, hipStream_t st);

}  // namespace gemm_impl
