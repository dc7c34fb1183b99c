// Shared helpers of the gated delta rule kernels (K16).
#pragma once
#include "ssm.h"

__device__ __forceinline__ float sigmoid_f32(float z) { return 1.0f / (1.0f + expf(-z)); }
// what norm and gate of a head's outputs make of one of them: its root and division as in mv_delta_step; in 16 bits the gate by hardware exponential and
// reciprocal (1 ulp of fp32 each)
__device__ __forceinline__ float head_rms(float squares, int channels, float eps, float out_scale) { return out_scale / sqrtf(squares / (float)channels + eps); }
__device__ __forceinline__ float gate_16(float z, int kind) {
  return (kind == MV_GATE_SIGMOID ? 1.f : z) * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
}
// log of the decay factor: -exp(a_log) * softplus(a + bias)
__device__ __forceinline__ float decay_log(float rate, float a, float bias) { return -rate * softplus_f32(a + bias); }

// chunked form (16-bit); MV_E_SHAPE when it does not apply
size_t mv_delta_chunk_workspace(int n_seqs, int total_q, int heads, int p, int n);
size_t mv_delta_segments_workspace(int n_seqs, int total_q, int max_q, int heads, int p, int n);   // beside it, where sequences are cut
// `normed` (NULL: not asked for): in: norm and gate in the walk whatever the rule on sizes says; out: they are already in the output
// `raw` (mv_delta_chunk_takes_conv): the channels ahead of the convolution, which goes to a.x if the walk reads it
int mv_delta_chunk_launch(const MvDeltaArgs &a, const void *raw, int64_t raw_stride, int dtype, bool *normed, hipStream_t stream);
bool mv_delta_chunk_takes_conv(const MvDeltaArgs &a, int dtype);
int mv_delta_scalar_launch(const MvDeltaArgs &a, const void *raw, int64_t raw_stride, bool *normed, hipStream_t stream);   // (from the above: bf16, one decay per head)
