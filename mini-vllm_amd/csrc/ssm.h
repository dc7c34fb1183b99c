// Shared helpers of the state space kernels (K15).
#pragma once
#include "latent.h"

__device__ __forceinline__ float silu_f32(float z) { return z / (1.0f + expf(-z)); }
// 16-bit operands: hardware exponential and reciprocal (1 ulp of fp32 each)
template <typename Tag>
__device__ __forceinline__ float silu_of(float z) {
  if constexpr (__is_same(Tag, f32_tag)) return silu_f32(z);
  else return z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
}
__device__ __forceinline__ float softplus_f32(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }

int mv_check_conv(const MvSsmArgs *a, int dtype);   // what mv_causal_conv refuses

// chunked form (16-bit); MV_E_SHAPE when it does not apply.  Without the workspace sequences are not cut into segments
size_t mv_ssm_chunk_workspace(int n_seqs, int total_q, int max_q, int heads, int p, int n);
int mv_ssm_chunk_launch(const MvSsmArgs &a, void *workspace, size_t ws_bytes, int total_q, int dtype, hipStream_t stream);
bool mv_ssm_chunk_cuts(int n_seqs, int total_q, int max_q, int heads, int p, int n);   // into segments
// the same for heads of 64 columns that share b and c
size_t mv_ssm_heads_workspace(int n_seqs, int total_q, int max_q, int heads, int p, int n);
int mv_ssm_heads_launch(const MvSsmArgs &a, void *workspace, size_t ws_bytes, int total_q, int dtype, hipStream_t stream);
