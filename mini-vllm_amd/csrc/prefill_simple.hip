// K2 (generic path) — packed varlen causal prefill attention on the vector
// ALU.  One wave per (query token, query head); keys are streamed exactly
// like the decode kernel does (LPT lanes per key row, online softmax per lane
// group).  This is the path of shapes that the MFMA kernels (prefill_mfma.hip,
// prefill_f32.hip: D in {64,128}) do not cover.
// Reference: minivllm/models/layers/attention.py:467-504,554-597.
#include "prefill_row.h"

namespace {

template <typename Tag, int D>
__global__ void __launch_bounds__(256) prefill_simple_kernel(PrefillParams p) {
  const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);  // (token, head)
  const int64_t total_q = p.cu_q[p.n_seqs];
  if (item >= total_q * p.n_heads) return;
  const int tok = (int)(item / p.n_heads);
  const int h = (int)(item - (int64_t)tok * p.n_heads);
  // which sequence owns this token (n_seqs is small: linear scan)
  int seq = 0;
  while (seq + 1 < p.n_seqs && p.cu_q[seq + 1] <= tok) ++seq;
  prefill_row<Tag, D>(p, seq, tok, h);
}

}  // namespace

int mv_prefill_simple_launch(const PrefillParams &p, int64_t max_total_q, int dtype, hipStream_t stream) {
  const int64_t items = max_total_q * p.n_heads;
  if (items == 0) return MV_OK;
  const unsigned blocks = (unsigned)((items + 3) / 4);
  if (p.head_dim == 256) {
    MV_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((prefill_simple_kernel<Tag, 256>), dim3(blocks), dim3(256), 0, stream, p));
  } else if (p.head_dim == 128) {
    MV_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((prefill_simple_kernel<Tag, 128>), dim3(blocks), dim3(256), 0, stream, p));
  } else if (p.head_dim == 64) {
    MV_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((prefill_simple_kernel<Tag, 64>), dim3(blocks), dim3(256), 0, stream, p));
  } else {
    return MV_E_SHAPE;
  }
  MV_LAUNCH_CHECK();
  return MV_OK;
}
