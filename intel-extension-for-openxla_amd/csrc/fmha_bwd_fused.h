// Interface of the fused attention backward kernels (fmha_bwd_fused.hip) for the entry point in
// fmha_bwd.hip.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace fmha_bwd_fused {

struct Args {
  const void* q;
  const void* k;
  const void* v;
  const void* d_o;
  const void* o;         // [units, F, H] output of the forward pass
  const void* bias;      // [units, F, T] additive bias or null
  const float* lse_fwd;  // [units, F] log-sum-exp of the forward pass
  float* lse;            // scratch [units, F]: LSE times log2(e)       } written by the queries-own launch,
  float* dsum;           // scratch [units, F]: D = rowsum(dO o O)       } read by the keys-own launches after it
  void* dq;
  void* dk;
  void* dv;
  int H, F, T;
  float scale;
  bool causal;
  bool stats_ready;      // lse and dsum have been formed; required where one_grid() says so
  void* ds;              // scratch for dS of ds_units units (saved_bytes()), or null: dS is formed again where it is needed
  uint64_t ds_units;
};

// Head sizes up to 256 (multiples of 8); a bias of at most 2 GiB per unit.
bool eligible(const Args& a, uint64_t units);
// Whether all passes should run as one grid, on statistics that are formed before it.
bool one_grid(const Args& a, uint64_t units);
// How many units' dS to keep at a time in `bytes` of scratch (0: keep none; H, F, T, causal and the presence of a bias of `a`).
uint64_t saved_units(const Args& a, uint64_t units, uint64_t bytes);
// Bytes in which `units` units keep dS (H, F, T and causal of `a`).
size_t saved_bytes(const Args& a, uint64_t units);
// Queries own (dQ; it also forms the two per-row statistics), then keys own (dK, dV).
void launch(const Args& a, uint64_t units, bool bf16, hipStream_t stream);

}  // namespace fmha_bwd_fused
