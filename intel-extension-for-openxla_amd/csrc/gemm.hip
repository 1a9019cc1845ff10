// bf16 / fp16 GEMM with fp32 accumulation and a fused epilogue:
//     out = act(alpha * op(lhs) op(rhs) + beta * c + bias)
//
// MFMA kernel (gemm_mfma_kernel): one work-group owns a BM x BN tile of the output and walks K in
// steps of BK (32 for the 256x256 tile, 64 for the smaller ones).  Operand tiles go from global memory
// straight into LDS (buffer_load ... lds, 16 bytes per lane, no staging registers and no ds_write): a
// wave's load fills 1 KiB of contiguous LDS, and the per-lane *global* address is chosen so that the
// data lands swizzled.  A ring of three or four LDS stages; the loads of later K steps are issued
// between the MFMAs of step t and are waited for with a counted s_waitcnt at the one barrier per step.
//   "KC" operand (reduction index contiguous in memory: A[M,K] row-major, B stored [N,K]):
//       LDS [row][64 k], the 16-byte chunks of a row XOR-swizzled by the row number, read
//       with one ds_read_b128 per fragment.
//   "MC" operand (free index contiguous: B[K,N] row-major, A stored [K,M]):
//       LDS [k][cols], chunks XOR-swizzled by k, read with the LDS transpose loads
//       (ds_read_b64_tr_b16), which hand each lane four consecutive k of one column.
// The products are issued with the operands swapped (D^T = B^T A^T) so that a lane ends up
// holding four consecutive output columns of one row.
//
// 16-bit operands whose strides or sizes the direct loads cannot take and all fp32 operands run gemm_ragged_kernel
// (gemm_ragged.h; fp32 on the large tile gemm_split_kernel, gemm_split.h), products of few tiles gemm_slices_kernel
// (gemm_slices.h), int8 operands the int8 MFMA kernel (gemm_s8.hip); what is left (operands of less than 16 bytes, int8
// products into an unaligned output) runs gemm_generic_kernel, a plain LDS-tiled kernel.  This is where the reference
// falls back to oneDNN (onednn_matmul_utils.cc:394-491).
#include <algorithm>

#include "gemm_kernel.h"
#include "gemm_ragged.h"
#include "gemm_rows.h"
#include "gemm_s8.h"
#include "gemm_slices.h"

namespace {

using namespace gemm_impl;

// ------------------------------------------------------------------ generic kernel
// Any accepted dtype triple, any strides/transposes: 16x16 threads, 64x64 tile,
// operands converted to fp32 (or int32) while staging.
enum : int { G_BF16 = 0, G_F16 = 1, G_F32 = 2, G_S8 = 3, G_S32 = 4 };

__device__ __forceinline__ float load_as_f32(const void* p, int kind, int64_t i) {
  switch (kind) {
    case G_BF16: return (float)reinterpret_cast<const __bf16*>(p)[i];
    case G_F16: return (float)reinterpret_cast<const _Float16*>(p)[i];
    case G_S8: return (float)reinterpret_cast<const int8_t*>(p)[i];
    case G_S32: return (float)reinterpret_cast<const int32_t*>(p)[i];
    default: return reinterpret_cast<const float*>(p)[i];
  }
}

struct GenericParams {
  const void* a;
  const void* b;
  void* out;
  const void* c;
  const void* bias;
  int M, N, K;
  int64_t lda, ldb, ldc, sa, sb, sc;
  int ta, tb;  // operand is the transpose of the stored matrix
  int kin, kout;
  float alpha, beta;
  int act;
  void* out_alt[2];  // see GemmParams
  int64_t sbias;
};

__global__ __launch_bounds__(256) void gemm_generic_kernel(GenericParams p) {
  __shared__ float As[16][65];
  __shared__ float Bs[16][65];
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  const int64_t bz = blockIdx.z;
  if (p.out_alt[0] && bz > 0) p.out = p.out_alt[bz - 1];
  const bool integer = p.kin == G_S8;
  float acc[4][4] = {};
  int iacc[4][4] = {};
  for (int k0 = 0; k0 < p.K; k0 += 16) {
    for (int e = threadIdx.x; e < 16 * 64; e += 256) {
      const int kk = e / 64, r = e % 64;
      const int k = k0 + kk;
      float av = 0.f, bv = 0.f;
      if (k < p.K && m0 + r < p.M) {
        const int64_t i = bz * p.sa + (p.ta ? (int64_t)k * p.lda + (m0 + r) : (int64_t)(m0 + r) * p.lda + k);
        av = load_as_f32(p.a, p.kin, i);
      }
      if (k < p.K && n0 + r < p.N) {
        const int64_t i = bz * p.sb + (p.tb ? (int64_t)(n0 + r) * p.ldb + k : (int64_t)k * p.ldb + (n0 + r));
        bv = load_as_f32(p.b, p.kin, i);
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
      if (integer) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) iacc[i][j] += (int)a[i] * (int)b[j];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= p.M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n >= p.N) continue;
      const int64_t off = bz * p.sc + (int64_t)m * p.ldc + n;
      if (integer) {
        reinterpret_cast<int32_t*>(p.out)[off] = iacc[i][j];
        continue;
      }
      float v = p.alpha * acc[i][j];
      if (p.beta != 0.f && p.c) v += p.beta * load_as_f32(p.c, p.kout, off);
      if (p.bias) v += load_as_f32(p.bias, p.kin, bz * p.sbias + n);
      v = apply_act(v, p.act);
      switch (p.kout) {
        case G_BF16: reinterpret_cast<__bf16*>(p.out)[off] = (__bf16)v; break;
        case G_F16: reinterpret_cast<_Float16*>(p.out)[off] = (_Float16)v; break;
        default: reinterpret_cast<float*>(p.out)[off] = v; break;
      }
    }
  }
}

// Second pass of a K-split GEMM: out = act(alpha * sum_z partial[z] + beta * c + bias), one rounding.
// partial: fp32 [ks][M][N], slices `stride` elements apart; out / c: [M][ldc] of kind kout; bias of kind kin.
struct ReduceParams {
  const float* partial;
  void* out;
  const void* c;
  const void* bias;
  int M, N, ks;
  int64_t stride;  // a multiple of 4
  int64_t ldc;
  int kin, kout;
  float alpha, beta;
  int act;
};
// What bounds it: one chain of latencies, arguments - loads - store, in a launch of a few work-groups.  So everything is asked for
// before the first sum, and the division that finds the row is one of 32 bits (a 64-bit division in front of a loop that waited for
// each slice in turn: 20 x 336 x 4808 11.5 -> 8.2 us for both launches, 290 x 128 x 10624 15.0 -> 11.1, 4 x 4096 x 16384 29.7 -> 29.3).
constexpr int kReduceAhead = 16;  // slices in flight together; the planner takes no more
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(ReduceParams p) {
  const int64_t idx = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;  // four consecutive elements of the packed product
  const int64_t total = (int64_t)p.M * p.N;
  if (idx >= total) return;
  floatx4 part[kReduceAhead];
#pragma unroll
  for (int z = 0; z < kReduceAhead; ++z)
    if (z < p.ks) part[z] = *reinterpret_cast<const floatx4*>(p.partial + z * p.stride + idx);
  int m, n;
  if (total <= 0xffffffffll) {  // (uniform)
    m = (int)((uint32_t)idx / (uint32_t)p.N);
    n = (int)((uint32_t)idx - (uint32_t)m * (uint32_t)p.N);
  } else {
    m = (int)(idx / p.N);
    n = (int)(idx % p.N);
  }
  const int count = (int)min((int64_t)4, total - idx);
  int64_t off[4];
  float add[4], cv[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {  // (past the end: the last element again)
    off[j] = (int64_t)m * p.ldc + n;
    add[j] = p.bias ? load_as_f32(p.bias, p.kin, n) : 0.f;
    cv[j] = p.beta != 0.f && p.c ? load_as_f32(p.c, p.kout, off[j]) : 0.f;
    if (j + 1 < count && ++n == p.N) { n = 0; ++m; }
  }
  floatx4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int z = 0; z < kReduceAhead; ++z)
    if (z < p.ks) s += part[z];
  for (int z = kReduceAhead; z < p.ks; ++z) s += *reinterpret_cast<const floatx4*>(p.partial + z * p.stride + idx);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (j >= count) break;
    float v = p.alpha * s[j];
    if (p.beta != 0.f && p.c) v += p.beta * cv[j];
    if (p.bias) v += add[j];
    v = apply_act(v, p.act);
    switch (p.kout) {
      case G_BF16: reinterpret_cast<__bf16*>(p.out)[off[j]] = (__bf16)v; break;
      case G_F16: reinterpret_cast<_Float16*>(p.out)[off[j]] = (_Float16)v; break;
      default: reinterpret_cast<float*>(p.out)[off[j]] = v; break;
    }
  }
}

// Copies operands whose rows start anywhere into rows of whole, aligned 16-byte chunks, zeros behind a row's end.
struct PackOperand {
  const uint16_t* from;
  uint16_t* to;
  int64_t ld_from, ld_to;
  int cols, row_chunks;  // chunks of eight elements
  int chunks;            // in all
};
constexpr int kPackPerThread = 4;
__global__ __launch_bounds__(256) void gemm_pack_kernel(PackOperand a, PackOperand b, int a_blocks) {
  const bool second = (int)blockIdx.x >= a_blocks;
  const PackOperand& p = second ? b : a;
  const int first = ((int)blockIdx.x - (second ? a_blocks : 0)) * 256 * kPackPerThread + (int)threadIdx.x;
  u32x4 v[kPackPerThread];
  uint16_t* to[kPackPerThread];
#pragma unroll
  for (int i = 0; i < kPackPerThread; ++i) {
    const int chunk = first + 256 * i;
    to[i] = nullptr;
    if (chunk >= p.chunks) continue;
    const int row = (int)((uint32_t)chunk / (uint32_t)p.row_chunks), col = (chunk - row * p.row_chunks) * 8;
    const uint16_t* from = p.from + row * p.ld_from + col;
    to[i] = p.to + row * p.ld_to + col;
    if (col + 8 <= p.cols) {
      __builtin_memcpy(&v[i], from, 16);
    } else {
      uint16_t e[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) e[j] = col + j < p.cols ? from[j] : (uint16_t)0;
      __builtin_memcpy(&v[i], e, 16);
    }
  }
#pragma unroll
  for (int i = 0; i < kPackPerThread; ++i)
    if (to[i]) *reinterpret_cast<u32x4*>(to[i]) = v[i];
}

// ------------------------------------------------------------------ host side

int generic_kind(int dtype) {
  switch (dtype) {
    case XMK_BF16: return G_BF16;
    case XMK_F16: return G_F16;
    case XMK_F32: return G_F32;
    case XMK_S8: return G_S8;
    case XMK_S32: return G_S32;
    default: return -1;
  }
}

int elem_size(int dtype) {
  switch (dtype) {
    case XMK_BF16: case XMK_F16: return 2;
    case XMK_F32: case XMK_S32: return 4;
    case XMK_S8: return 1;
    default: return 0;
  }
}

// What runs a policy's tile: the kernels that take any alignment have names of their own.
const char* kernel_name(int policy, bool any_alignment) {
  if (!any_alignment || is_slices(policy)) return kPolicies[policy].name;
  return kPolicies[policy].bm == 128 ? "ragged_128x128" : "ragged_64x64";
}
// Whether an operand is long enough for the loaders of those kernels, which read 16 bytes at a time.
bool spans_a_load(int64_t rows, int64_t ld, int64_t cols, int dtype) { return ((rows - 1) * ld + cols) * elem_size(dtype) >= 16; }

}  // namespace

extern "C" const char* xmk_gemm_policy_name(int64_t m, int64_t n, int64_t k, int32_t rhs_transpose,
                                            int32_t dtype_in, int32_t dtype_out) {
  const bool sixteen = dtype_in == XMK_BF16 || dtype_in == XMK_F16, f32 = dtype_in == XMK_F32;
  if (dtype_in == XMK_S8 && dtype_out == XMK_S32) return "mfma_s8_128x128x64";
  if (!(sixteen || f32) || !(dtype_out == dtype_in || dtype_out == XMK_F32)) return "generic_64x64";
  // (packed operands at aligned addresses assumed, as everywhere in this query)
  const bool any_alignment = f32 || k % 8 != 0 || (!rhs_transpose && n % 8 != 0);
  if (any_alignment && !(spans_a_load(m, k, k, dtype_in) && spans_a_load(k, n, n, dtype_in))) return "generic_64x64";
  const int cls = f32 ? kClassF32 : any_alignment ? kClassRagged : rhs_transpose ? kClassNK : kClassKN;
  int rows_kind = kRowsNone;
  if (sixteen && m >= 1 && m <= kRowsMaxM && k % 8 == 0) {
    if (!rhs_transpose && n % 8 == 0) rows_kind = kRowsMC;
    if (rhs_transpose && k <= kColsMaxK) rows_kind = kRowsKC;
  }
  return kernel_name(select_policy(m, n, k, 1, rows_kind, cls, false), any_alignment);
}

namespace {
// out1 / out2: further outputs of the shared-lhs three-GEMM form, or null for a plain GEMM.
// policy: tile policy to use instead of select_policy's choice (the K-split planner's), or -1.
// kslice: K slice of a batch member (a K split into unequal slices; the operands are then those of the whole
// product), or 0.
// padded: the operands' rows hold whole 16-byte chunks, whatever their lengths.
int run_gemm(const xmk_gemm_desc* d, void* out1, void* out2, void* stream, int policy = -1, int kslice = 0, bool padded = false);

// The tile loaders form byte offsets of up to 256 rows of an operand in 32 bits.
constexpr int64_t kMaxLd = int64_t{1} << 22;

// The conditions of the direct-to-LDS 16-bit kernels on the stored operands.
bool direct_ok(const xmk_matrix& lhs, const xmk_matrix& rhs, bool padded = false) {
  return xmk::aligned(lhs.data, 16) && xmk::aligned(rhs.data, 16) && lhs.leading_dim_stride % 8 == 0 &&
         rhs.leading_dim_stride % 8 == 0 && lhs.batch_stride % 8 == 0 && rhs.batch_stride % 8 == 0 &&
         (padded || (lhs.num_cols % 8 == 0 && rhs.num_cols % 8 == 0));
}

// Which streaming kernel for a few rows (gemm_rows.hip) can run this descriptor's product, if any.
int rows_kind_desc(const xmk_gemm_desc* d, int64_t m, int64_t n, int64_t k) {
  if (d->out.transpose || d->lhs.transpose || !direct_ok(d->lhs, d->rhs) || !xmk::aligned(d->out.data, 16))
    return kRowsNone;
  if (d->dtype_in != XMK_BF16 && d->dtype_in != XMK_F16) return kRowsNone;
  GemmParams p{};
  p.M = (int)m; p.N = (int)n; p.K = (int)k;
  p.lda = d->lhs.leading_dim_stride; p.ldb = d->rhs.leading_dim_stride;
  return gemm_rows_applicable(p, false, d->rhs.transpose == 0);
}

// K slices worth using for a plain 16-bit GEMM of this shape when scratch is available: few
// output tiles (the device has 256 CUs) and a long reduction.  1: do not split.
// *policy: the tile policy of the slices (-1: whatever select_policy picks for a slice).
// *kslice: K slice (a multiple of 64, the last slice takes the rest) of operands passed whole, 0: equal slices as batch members.
int plan_splitk(const xmk_gemm_desc* d, int64_t m, int64_t n, int64_t k, int* policy, int* kslice, bool padded = false) {
  *policy = -1;
  *kslice = 0;
  if (d->batch_size != 1) return 1;
  if (d->dtype_in != XMK_BF16 && d->dtype_in != XMK_F16 && d->dtype_in != XMK_F32) return 1;
  // XMK_GEMM_SPLITK=<slices> overrides the choice (read at every call; the autotuner's handle).
  const char* forced_env = getenv("XMK_GEMM_SPLITK");
  const int forced = forced_env ? atoi(forced_env) : 0;
  if (d->dtype_in == XMK_F32 || !direct_ok(d->lhs, d->rhs, padded)) {
    Choice c = cheapest(m, n, k, 1, d->dtype_in == XMK_F32 ? kClassF32 : kClassRagged, true);
    if (forced >= 1) c.slices = forced;
    if (forced_policy() >= 0) c.policy = forced_policy();
    if (c.slices < 2) return 1;
    *policy = c.policy;
    *kslice = (int)(xmk::ceil_div(xmk::ceil_div(k, c.slices), 64) * 64);
    return (int)xmk::ceil_div(k, *kslice);
  }
  auto divides = [&](int ks) { return ks >= 1 && ks <= 16 && k % (ks * 8) == 0; };
  if (forced >= 1) return divides(forced) ? forced : 1;
  const int rows_kind = (forced_policy() < 0 || forced_policy() == kRowsPolicy) ? rows_kind_desc(d, m, n, k) : kRowsNone;
  const bool rows_ok = rows_kind != kRowsNone;
  // (the table was measured with B stored [K, N])
  if (const TunedShape* t = tuned_shape(m, n, k); forced_policy() == kUnforced && !d->rhs.transpose && t && t->ksplit >= 1 &&
                                                  divides(t->ksplit) && (t->policy != kRowsPolicy || rows_ok)) {
    if (t->ksplit > 1) *policy = t->policy;
    return t->ksplit;
  }
  if (rows_streams_by_default(rows_kind, m, n)) return 1;  // streamed in one launch
  if (rows_ok && forced_policy() == kRowsPolicy) {
    // The streaming kernel forced on a narrower matrix (tests, the autotuner): slices until its narrowest
    // column blocks are about one work-group per CU, each slice keeping 512 rows (a batch of 64 per wave).
    const int64_t blocks = xmk::ceil_div(n, (int64_t)(rows_kind == kRowsMC ? kRowsMinBN : kColsBN));
    int ks = 1;
    if (blocks < kRowsEnoughBlocks)
      while (ks < 16 && blocks * ks < 256 && k % (ks * 2 * 8) == 0 && k / (ks * 2) >= 512) ks *= 2;
    if (ks > 1) *policy = kRowsPolicy;
    return ks;
  }
  const Choice c = cheapest(m, n, k, 1, d->rhs.transpose ? kClassNK : kClassKN, true);
  if (c.slices < 2) return 1;
  *policy = c.policy;
  if (k % (8 * c.slices) == 0) return c.slices;
  // Equal slices would not start on 16 bytes: slices of whole K steps, the last one shorter.  (Such k went without a split:
  // 64 x 4096 x 9752 75.7 -> 29.3 us, 128 x 1024 x 8200 37.2 -> 14.4, 256 x 512 x 12296 50.5 -> 17.8.)
  *kslice = (int)(xmk::ceil_div(xmk::ceil_div(k, c.slices), 64) * 64);
  return (int)xmk::ceil_div(k, *kslice);
}

// Elements from one slice's partial sums to the next (16-byte aligned).
int64_t slice_stride(int64_t m, int64_t n) { return (m * n + 3) / 4 * 4; }

void gemm_dims(const xmk_gemm_desc* d, int64_t* m, int64_t* n, int64_t* k) {
  const bool t = d->out.transpose != 0;  // C^T = B^T A^T swaps the roles
  const xmk_matrix& lhs = t ? d->rhs : d->lhs;
  const xmk_matrix& rhs = t ? d->lhs : d->rhs;
  const bool lt = t ? !lhs.transpose : lhs.transpose, rt = t ? !rhs.transpose : rhs.transpose;
  *m = lt ? lhs.num_cols : lhs.num_rows;
  *k = lt ? lhs.num_rows : lhs.num_cols;
  *n = rt ? rhs.num_rows : rhs.num_cols;
}
}  // namespace

extern "C" int xmk_gemm(const xmk_gemm_desc* d, void* stream) { return run_gemm(d, nullptr, nullptr, stream); }

namespace {
// The K slices that a call with scratch runs this descriptor's product in (see plan_splitk); 1: scratch is not used.
int planned_slices(const xmk_gemm_desc* d, int64_t* m, int64_t* n, int64_t* k, int* policy, int* kslice, bool padded = false) {
  if (d->lhs.transpose || d->out.transpose) return 1;
  gemm_dims(d, m, n, k);
  if (*m <= 0 || *n <= 0 || *k <= 0) return 1;
  return plan_splitk(d, *m, *n, *k, policy, kslice, padded);
}

// Whether run_gemm would take the product (untransposed lhs and output): the scratch paths hand it other operands, and what it
// would have rejected must still be rejected (a reduction size that differs between the operands, a leading dimension
// shorter than the full row).
bool valid_product(const xmk_gemm_desc* d, int* act, bool* wants_bias) {
  *act = ACT_NONE;
  *wants_bias = false;
  switch (d->epilogue) {
    case XMK_EPI_DEFAULT: break;
    case XMK_EPI_RELU: *act = ACT_RELU; break;
    case XMK_EPI_GELU: *act = ACT_GELU; break;
    case XMK_EPI_BIAS: *wants_bias = true; break;
    case XMK_EPI_BIAS_RELU: *wants_bias = true; *act = ACT_RELU; break;
    case XMK_EPI_BIAS_GELU: *wants_bias = true; *act = ACT_GELU; break;
    default: return false;
  }
  int64_t m, n, k;
  gemm_dims(d, &m, &n, &k);
  const int64_t k_rhs = d->rhs.transpose ? d->rhs.num_cols : d->rhs.num_rows;
  if (k_rhs != k || d->lhs.leading_dim_stride < d->lhs.num_cols || d->rhs.leading_dim_stride < d->rhs.num_cols) return false;
  return !((*wants_bias && !d->bias) || (d->beta != 0.0f && !d->c) || !d->out.data || d->out.num_rows != m || d->out.num_cols != n ||
           d->out.leading_dim_stride < n || (d->dtype_out != d->dtype_in && d->dtype_out != XMK_F32));
}

// Copying operands with misaligned rows into scratch first, for the direct-to-LDS kernels: a load at an unaligned address
// takes the CU's load path as long as four, and a large product makes every such load tens of times, the copy once.
// Microseconds without / with the copy: 1023 x 5003 x 2047 55.7 / 43, 4001^3 197 / 142, 1418 x 8367 x 3357 176 / 114, 2047^3
// 37 / 32; 64 x 5001 x 5001 23.5 / 34, 300 x 50257 x 769 65 / 101: chosen by the estimates of both ways.  The second one's: the
// direct kernels' on aligned sizes, what the copy takes (fitted to 51 odd sizes: 5.2 us and 0.165 per MB) and what outputs of
// odd row length cost beyond aligned ones (0.87 per million).  On those 51 it never chose the slower way.
struct PackPlan {
  bool a, b;             // which are copied
  int64_t lda, ldb;      // leading dimensions of the copies
  size_t b_at, total;    // bytes
};
bool plan_pack(const xmk_gemm_desc* d, PackPlan* p) {
  if (d->lhs.transpose || d->out.transpose || d->batch_size != 1) return false;
  if (d->dtype_in != XMK_BF16 && d->dtype_in != XMK_F16) return false;
  if (direct_ok(d->lhs, d->rhs) || !xmk::aligned(d->out.data, 16)) return false;
  auto ok = [](const xmk_matrix& x) { return xmk::aligned(x.data, 16) && x.leading_dim_stride % 8 == 0 && x.num_cols % 8 == 0; };
  auto ld = [](const xmk_matrix& x) { return xmk::ceil_div(x.num_cols, 64) * 64; };
  int64_t m, n, k;
  gemm_dims(d, &m, &n, &k);
  constexpr int64_t kMax = 1 << 29;
  if (m <= 0 || n <= 0 || k <= 0 || m >= kMax || n >= kMax || k >= kMax || m * k >= kMax || n * k >= kMax) return false;
  p->a = !ok(d->lhs);
  p->b = !ok(d->rhs);
  if (!p->a && !p->b) return false;  // (only a batch stride, of a single member, is no multiple of eight)
  p->lda = ld(d->lhs);
  p->ldb = ld(d->rhs);
  if ((p->a && p->lda >= kMaxLd) || (p->b && p->ldb >= kMaxLd)) return false;  // (rows of just under 2^22 are taken as they are)
  p->b_at = p->a ? (size_t)m * p->lda * 2 : 0;
  p->total = p->b_at + (p->b ? (size_t)d->rhs.num_rows * p->ldb * 2 : 0);
  if (forced_policy() != kUnforced || getenv("XMK_GEMM_SPLITK")) return false;  // (they force what runs on the operands given)
  if (!spans_a_load(m, d->lhs.leading_dim_stride, k, d->dtype_in) ||
      !spans_a_load(d->rhs.num_rows, d->rhs.leading_dim_stride, d->rhs.num_cols, d->dtype_in)) return false;
  const float copied = (float)((p->a ? m * k : 0) + (p->b ? n * k : 0)) * 2e-6f;
  const float with = cheapest(m, n, k, 1, d->rhs.transpose ? kClassNK : kClassKN, true).us + 5.2f + 0.165f * copied + 0.87e-6f * (float)m * (float)n;
  return cheapest(m, n, k, 1, kClassRagged, true).us > 1.03f * with;
}
// The descriptor with the copies at `ws` in place of the operands.
xmk_gemm_desc packed_desc(const xmk_gemm_desc* d, const PackPlan& p, char* ws) {
  xmk_gemm_desc q = *d;
  q.lhs.batch_stride = q.rhs.batch_stride = 0;  // (one member: nothing is a stride away from it)
  if (p.a) { q.lhs.data = ws; q.lhs.leading_dim_stride = p.lda; }
  if (p.b) { q.rhs.data = ws + p.b_at; q.rhs.leading_dim_stride = p.ldb; }
  return q;
}
PackOperand pack_operand(const xmk_matrix& x, void* to, int64_t ld) {
  PackOperand p{};
  p.from = (const uint16_t*)x.data; p.to = (uint16_t*)to; p.ld_from = x.leading_dim_stride; p.ld_to = ld;
  p.cols = (int)x.num_cols; p.row_chunks = (int)xmk::ceil_div(x.num_cols, 8); p.chunks = (int)(x.num_rows * p.row_chunks);
  return p;
}
int gemm_ws(const xmk_gemm_desc* d, void* workspace, size_t workspace_bytes, void* stream, bool padded);
}  // namespace

extern "C" size_t xmk_gemm_workspace_bytes(const xmk_gemm_desc* d) {
  if (!d) return 0;
  int64_t m, n, k;
  int policy, kslice;
  const int ks = planned_slices(d, &m, &n, &k, &policy, &kslice);
  const size_t need = ks > 1 ? (size_t)ks * slice_stride(m, n) * sizeof(float) : 0;
  PackPlan pk;
  if (!plan_pack(d, &pk)) return need;
  const xmk_gemm_desc q = packed_desc(d, pk, nullptr);
  const int kp = planned_slices(&q, &m, &n, &k, &policy, &kslice, true);
  return std::max(need, pk.total + (kp > 1 ? (size_t)kp * slice_stride(m, n) * sizeof(float) : 0));
}

extern "C" int xmk_gemm_ws(const xmk_gemm_desc* d, void* workspace, size_t workspace_bytes, void* stream) {
  if (!d) return xmk::fail(XMK_INVALID_ARGUMENT, "gemm: null descriptor");
  if (!workspace || !xmk::aligned(workspace, 16)) return run_gemm(d, nullptr, nullptr, stream);
  PackPlan pk;
  int act;
  bool wants_bias;
  if (plan_pack(d, &pk) && pk.total <= workspace_bytes && d->lhs.data && d->rhs.data && d->lhs.leading_dim_stride < kMaxLd &&
      d->rhs.leading_dim_stride < kMaxLd && d->out.leading_dim_stride < kMaxLd && valid_product(d, &act, &wants_bias)) {
    const xmk_gemm_desc q = packed_desc(d, pk, (char*)workspace);
    PackOperand a{}, b{};
    if (pk.a) a = pack_operand(d->lhs, workspace, pk.lda);
    if (pk.b) b = pack_operand(d->rhs, (char*)workspace + pk.b_at, pk.ldb);
    auto blocks = [](const PackOperand& p) { return (int)xmk::ceil_div(p.chunks, 256 * kPackPerThread); };
    xmk::trace("gemm: %s copied into aligned rows", pk.a && pk.b ? "both operands" : pk.a ? "lhs" : "rhs");
    hipLaunchKernelGGL(gemm_pack_kernel, dim3((unsigned)(blocks(a) + blocks(b))), dim3(256), 0, (hipStream_t)stream, a, b, blocks(a));
    return gemm_ws(&q, (char*)workspace + pk.total, workspace_bytes - pk.total, stream, true);
  }
  return gemm_ws(d, workspace, workspace_bytes, stream, false);
}

namespace {
int gemm_ws(const xmk_gemm_desc* d, void* workspace, size_t workspace_bytes, void* stream, bool padded) {
  int64_t m, n, k;
  int slice_policy, kslice;
  const int ks = planned_slices(d, &m, &n, &k, &slice_policy, &kslice, padded);
  if (ks < 2 || workspace_bytes < (size_t)ks * slice_stride(m, n) * sizeof(float))
    return run_gemm(d, nullptr, nullptr, stream, -1, 0, padded);
  // Pass 1: the K slices as a batched GEMM into fp32 partial sums (no epilogue); a slice is a
  // column range of lhs and a row (or column) range of rhs, so only the batch strides change.
  xmk_gemm_desc p = *d;
  if (!kslice) {
    const int64_t kz = k / ks;
    p.lhs.num_cols = kz;
    p.lhs.batch_stride = kz;
    if (p.rhs.transpose) { p.rhs.num_cols = kz; p.rhs.batch_stride = kz; }
    else { p.rhs.num_rows = kz; p.rhs.batch_stride = kz * p.rhs.leading_dim_stride; }
  }
  p.out.data = workspace; p.out.leading_dim_stride = n; p.out.batch_stride = slice_stride(m, n);
  p.c = nullptr; p.bias = nullptr;
  p.dtype_out = XMK_F32;
  p.batch_size = ks; p.alpha = 1.0f; p.beta = 0.0f; p.epilogue = XMK_EPI_DEFAULT;
  int act;
  bool wants_bias;
  if (!valid_product(d, &act, &wants_bias)) return run_gemm(d, nullptr, nullptr, stream);  // reports the error
  xmk::trace("gemm m=%lld n=%lld k=%lld -> split K %d ways", (long long)m, (long long)n, (long long)k, ks);
  int rc = run_gemm(&p, nullptr, nullptr, stream, slice_policy, kslice, padded);
  if (rc != XMK_OK) return rc;
  ReduceParams r;
  r.partial = (const float*)workspace; r.out = d->out.data; r.c = d->beta != 0.0f ? d->c : nullptr;
  r.bias = wants_bias ? d->bias : nullptr;
  r.M = (int)m; r.N = (int)n; r.ks = ks; r.stride = slice_stride(m, n); r.ldc = d->out.leading_dim_stride;
  r.kin = generic_kind(d->dtype_in); r.kout = generic_kind(d->dtype_out);
  r.alpha = d->alpha; r.beta = d->beta; r.act = act;
  hipLaunchKernelGGL(gemm_splitk_reduce_kernel, dim3((unsigned)xmk::ceil_div(m * n, 4 * 256)), dim3(256), 0,
                     (hipStream_t)stream, r);
  return xmk::check_launch("gemm");
}
}  // namespace

extern "C" int xmk_gemm_qkv(const xmk_gemm_desc* d, void* out_k, void* out_v, void* stream) {
  if (!d) return xmk::fail(XMK_INVALID_ARGUMENT, "gemm_qkv: null descriptor");
  if (!out_k || !out_v) return xmk::fail(XMK_INVALID_ARGUMENT, "gemm_qkv: null output");
  if (d->batch_size != 1 || d->beta != 0.0f || d->out.transpose)
    return xmk::fail(XMK_INVALID_ARGUMENT, "gemm_qkv: needs batch_size 1, beta 0 and a row-major output");
  if (d->dtype_in != d->dtype_out || (d->dtype_in != XMK_BF16 && d->dtype_in != XMK_F16))
    return xmk::fail(XMK_UNIMPLEMENTED, "gemm_qkv: 16-bit input and output of one type only");  // gemm.h:112-170
  return run_gemm(d, out_k, out_v, stream);
}

namespace {
int run_gemm(const xmk_gemm_desc* d, void* out1, void* out2, void* stream, int policy, int kslice, bool padded) {
  if (!d) return xmk::fail(XMK_INVALID_ARGUMENT, "gemm: null descriptor");
  if (!d->lhs.data || !d->rhs.data || !d->out.data)
    return xmk::fail(XMK_INVALID_ARGUMENT, "gemm: null operand");
  // Accepted dtype triples: onednn_matmul_utils.cc:605-610.
  const int din = d->dtype_in, dout = d->dtype_out;
  const bool ok_types = (din == XMK_BF16 && (dout == XMK_BF16 || dout == XMK_F32)) ||
                        (din == XMK_F16 && (dout == XMK_F16 || dout == XMK_F32)) ||
                        (din == XMK_F32 && dout == XMK_F32) || (din == XMK_S8 && dout == XMK_S32);
  if (!ok_types)
    return xmk::fail(XMK_INTERNAL, "Unexpected GEMM lhs type %d, rhs type %d and output type %d", din,
                     din, dout);
  int act = ACT_NONE;
  bool wants_bias = false;
  switch (d->epilogue) {
    case XMK_EPI_DEFAULT: break;
    case XMK_EPI_RELU: act = ACT_RELU; break;
    case XMK_EPI_GELU: act = ACT_GELU; break;
    case XMK_EPI_BIAS: wants_bias = true; break;
    case XMK_EPI_BIAS_RELU: wants_bias = true; act = ACT_RELU; break;
    case XMK_EPI_BIAS_GELU: wants_bias = true; act = ACT_GELU; break;
    case XMK_EPI_GELU_AUX:
    case XMK_EPI_BIAS_GELU_AUX:
      // onednn_matmul_utils.cc:321-322,452-453
      return xmk::fail(XMK_UNIMPLEMENTED, "Unsupported Activation mode");
    default: return xmk::fail(XMK_INTERNAL, "Unknown Epilogue.");
  }
  if (wants_bias && !d->bias)
    return xmk::fail(XMK_INVALID_ARGUMENT, "gemm: epilogue adds a vector bias but bias is null");
  if (d->beta != 0.0f && !d->c)
    return xmk::fail(XMK_INVALID_ARGUMENT, "gemm: beta != 0 but c is null");
  if (d->batch_size < 1) return xmk::fail(XMK_INVALID_ARGUMENT, "gemm: batch_size < 1");

  // Column-major output: C^T = B^T A^T (MakeBlasGemmCompatible, onednn_matmul_utils.cc:513-530).
  xmk_matrix lhs = d->lhs, rhs = d->rhs, out = d->out;
  if (out.transpose) {
    xmk_matrix t = lhs;
    lhs = rhs;
    rhs = t;
    lhs.transpose = !lhs.transpose;
    rhs.transpose = !rhs.transpose;
    out.transpose = 0;
  }
  const int64_t m = lhs.transpose ? lhs.num_cols : lhs.num_rows;
  const int64_t k = lhs.transpose ? lhs.num_rows : lhs.num_cols;
  const int64_t k2 = rhs.transpose ? rhs.num_cols : rhs.num_rows;
  const int64_t n = rhs.transpose ? rhs.num_rows : rhs.num_cols;
  if (m <= 0 || n <= 0 || k <= 0) return xmk::fail(XMK_INVALID_ARGUMENT, "gemm: empty dimension");
  if (k != k2)
    return xmk::fail(XMK_INVALID_ARGUMENT, "gemm: reduction sizes differ (lhs %lld, rhs %lld)",
                     (long long)k, (long long)k2);
  if (out.num_rows != m || out.num_cols != n)
    return xmk::fail(XMK_INVALID_ARGUMENT, "gemm: output is %lldx%lld, product is %lldx%lld",
                     (long long)out.num_rows, (long long)out.num_cols, (long long)m, (long long)n);
  if (lhs.leading_dim_stride < lhs.num_cols || rhs.leading_dim_stride < rhs.num_cols ||
      out.leading_dim_stride < n)
    return xmk::fail(XMK_INVALID_ARGUMENT, "gemm: leading_dim_stride smaller than the row length");
  if (m > INT32_MAX / 2 || n > INT32_MAX / 2 || k > INT32_MAX / 2 || d->batch_size > 65535)
    return xmk::fail(XMK_INVALID_ARGUMENT, "gemm: dimension too large");
  if (!d->bias && wants_bias) return xmk::fail(XMK_INVALID_ARGUMENT, "gemm: bias missing");
  if (lhs.leading_dim_stride >= kMaxLd || rhs.leading_dim_stride >= kMaxLd || out.leading_dim_stride >= kMaxLd)
    return xmk::fail(XMK_INVALID_ARGUMENT, "gemm: leading_dim_stride of 2^22 elements or more");

  hipStream_t st = (hipStream_t)stream;
  const bool qkv = out1 != nullptr;
  const bool sixteen = din == XMK_BF16 || din == XMK_F16;
  const bool fast = sixteen && direct_ok(lhs, rhs, padded) && xmk::aligned(out.data, 16) && xmk::aligned(out1, 16) &&
                    xmk::aligned(out2, 16);
  // 16-bit operands that miss those conditions and fp32 operands: the kernels that take any alignment (they read
  // 16 bytes at a time, wherever an operand has that many).
  auto spans = [&](const xmk_matrix& x) { return spans_a_load(x.num_rows, x.leading_dim_stride, x.num_cols, din); };
  const bool ragged = !fast && (sixteen || din == XMK_F32) && spans(lhs) && spans(rhs);
  if (fast || ragged) {
    GemmParams p;
    p.a = lhs.data; p.b = rhs.data; p.out = out.data; p.c = d->beta != 0.0f ? d->c : nullptr;
    p.bias = wants_bias ? d->bias : nullptr;
    p.M = (int)m; p.N = (int)n; p.K = (int)k;
    p.lda = lhs.leading_dim_stride; p.ldb = rhs.leading_dim_stride; p.ldc = out.leading_dim_stride;
    p.sa = lhs.batch_stride; p.sb = rhs.batch_stride; p.sc = out.batch_stride;
    p.alpha = d->alpha; p.beta = d->beta; p.act = act;
    p.out_alt[0] = out1; p.out_alt[1] = out2; p.sbias = 0;
    if (qkv) { p.sa = 0; p.sc = 0; p.sbias = n; }
    p.kslice = kslice;
    auto misaligned = [&](const xmk_matrix& x) {
      const int64_t size = elem_size(din);
      return !xmk::aligned(x.data, 16) || x.leading_dim_stride * size % 16 || x.batch_stride * size % 16;
    };
    p.misaligned = misaligned(lhs) || misaligned(rhs);
    if (kslice) { p.sa = 0; p.sb = 0; }
    const bool a_mc = lhs.transpose != 0;   // stored [K, M]
    const bool b_mc = rhs.transpose == 0;   // stored [K, N]
    const int batch = qkv ? 3 : (int)d->batch_size;
    const int rows_kind = fast ? gemm_rows_applicable(p, a_mc, b_mc) : kRowsNone;
    // the forced policy first, then the K-split planner's, then the table and the rules (three products that share
    // an operand take the tile one of them would: the results are then the same bits)
    const int pol = (forced_policy() < 0 && policy >= 0 && policy < kNumPolicies &&
                     (policy != kRowsPolicy || rows_kind != kRowsNone))
                        ? policy : select_policy(m, n, k, qkv ? 1 : batch, qkv ? kRowsNone : rows_kind,
                                        din == XMK_F32 ? kClassF32 : ragged ? kClassRagged : b_mc ? kClassKN : kClassNK, a_mc);
    xmk::trace("gemm m=%lld n=%lld k=%lld batch=%lld lhs_t=%d rhs_t=%d epilogue=%d beta=%g -> %s",
               (long long)m, (long long)n, (long long)k, (long long)d->batch_size, lhs.transpose,
               rhs.transpose, d->epilogue, d->beta, kernel_name(pol, ragged));
    // f(element type, fp32 output)
    auto typed = [&](auto&& f) {
      if (din == XMK_F32) f(float{}, std::true_type{});
      else if (din == XMK_BF16 && dout == XMK_F32) f(__bf16{}, std::true_type{});
      else if (din == XMK_BF16) f(__bf16{}, std::false_type{});
      else if (dout == XMK_F32) f(_Float16{}, std::true_type{});
      else f(_Float16{}, std::false_type{});
    };
    if (is_slices(pol)) {
      typed([&](auto t, auto o) { launch_slices<decltype(t), decltype(o)::value>(a_mc, b_mc, pol - kSlicesPolicy, p, batch, st); });
      return xmk::check_launch("gemm");
    }
    if (ragged) {
      typed([&](auto t, auto o) { launch_ragged<decltype(t), decltype(o)::value>(a_mc, b_mc, p, batch, kPolicies[pol].bm, st); });
      return xmk::check_launch("gemm");
    }
    if (pol == kRowsPolicy) {
      launch_gemm_rows(p, b_mc, din == XMK_BF16, dout == XMK_F32, batch, st);
      return xmk::check_launch("gemm");
    }
    if (din == XMK_BF16) {
      if (dout == XMK_F32) launch_layout<__bf16, true>(a_mc, b_mc, pol, p, batch, st);
      else launch_layout<__bf16, false>(a_mc, b_mc, pol, p, batch, st);
    } else {
      if (dout == XMK_F32) launch_layout<_Float16, true>(a_mc, b_mc, pol, p, batch, st);
      else launch_layout<_Float16, false>(a_mc, b_mc, pol, p, batch, st);
    }
    return xmk::check_launch("gemm");
  }

  if (din == XMK_S8 && (d->alpha != 1.0f || d->beta != 0.0f || d->epilogue != XMK_EPI_DEFAULT))
    return xmk::fail(XMK_UNIMPLEMENTED, "gemm: s8 x s8 -> s32 supports alpha=1, beta=0, no epilogue");
  if (din == XMK_S8 && dout == XMK_S32 && xmk::aligned(out.data, 16) && xmk::aligned(out1, 16) && xmk::aligned(out2, 16)) {
    GemmParams p{};
    p.a = lhs.data; p.b = rhs.data; p.out = out.data;
    p.M = (int)m; p.N = (int)n; p.K = (int)k;
    p.lda = lhs.leading_dim_stride; p.ldb = rhs.leading_dim_stride; p.ldc = out.leading_dim_stride;
    p.sa = lhs.batch_stride; p.sb = rhs.batch_stride; p.sc = out.batch_stride;
    p.out_alt[0] = out1; p.out_alt[1] = out2;
    if (qkv) { p.sa = 0; p.sc = 0; }
    auto vec16 = [](const xmk_matrix& x) {
      return (xmk::aligned(x.data, 16) && x.leading_dim_stride % 16 == 0 && x.batch_stride % 16 == 0 && x.num_cols % 16 == 0) ? 16 : 1;
    };
    p.vec_a = vec16(lhs);
    p.vec_b = vec16(rhs);
    xmk::trace("gemm m=%lld n=%lld k=%lld batch=%lld lhs_t=%d rhs_t=%d -> mfma_s8_128x128x64", (long long)m,
               (long long)n, (long long)k, (long long)d->batch_size, lhs.transpose, rhs.transpose);
    launch_gemm_s8(p, lhs.transpose != 0, rhs.transpose == 0, qkv ? 3 : (int)d->batch_size, st);
    return xmk::check_launch("gemm");
  }
  GenericParams g;
  g.a = lhs.data; g.b = rhs.data; g.out = out.data; g.c = d->beta != 0.0f ? d->c : nullptr;
  g.bias = wants_bias ? d->bias : nullptr;
  g.M = (int)m; g.N = (int)n; g.K = (int)k;
  g.lda = lhs.leading_dim_stride; g.ldb = rhs.leading_dim_stride; g.ldc = out.leading_dim_stride;
  g.sa = lhs.batch_stride; g.sb = rhs.batch_stride; g.sc = out.batch_stride;
  g.ta = lhs.transpose; g.tb = rhs.transpose;
  g.kin = generic_kind(din); g.kout = generic_kind(dout);
  g.alpha = d->alpha; g.beta = d->beta; g.act = act;
  g.out_alt[0] = out1; g.out_alt[1] = out2; g.sbias = 0;
  if (qkv) { g.sa = 0; g.sc = 0; g.sbias = n; }
  xmk::trace("gemm m=%lld n=%lld k=%lld -> generic_64x64", (long long)m, (long long)n, (long long)k);
  hipLaunchKernelGGL(gemm_generic_kernel,
                     dim3((unsigned)xmk::ceil_div(n, 64), (unsigned)xmk::ceil_div(m, 64),
                          (unsigned)(qkv ? 3 : d->batch_size)),
                     dim3(256), 0, st, g);
  return xmk::check_launch("gemm");
}
}  // namespace
