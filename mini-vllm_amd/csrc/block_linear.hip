// K20 — several projections with inputs and outputs of their own over the same rows (16-bit): out[:, block] = x[:, its inputs] W_block^T.
//
// For inputs of a low rank (64 or 128 channels): bound by the rows that it writes.  A workgroup takes 128 rows and 128 outputs of a block; its rows of x come
// by LDS-DMA at once (no step of channels follows another), four workgroups and more a CU cover that for each other.  A wave has 64 rows x 64 outputs
// and holds its part of W in registers.  W is the left operand, its rows dealt so that two tiles together give a lane eight outputs next to each other.
// 9939 rows, 2 x (128 -> 1024): 36 us by the library over the whole weight, half of it zeros; 21 with the rows of a tile one behind the other -> 19 with
// its outputs so (2.2 TB/s written: 1248 workgroups are two rounds of a few microseconds each); 16 000 rows 29 -> 27.
#include "latent.h"

namespace {

struct BlockLinear {
  MvBlockLinearArgs a;
  int tiles[MV_BLOCK_LINEAR_MAX], all;   // of outputs: of the blocks before, of all blocks
};
constexpr int BM = 128, BN = 128;

template <typename Tag, int KS>   // channels / 32
__global__ void __launch_bounds__(256, 4) block_linear_kernel(BlockLinear q) {
  typedef typename elem<Tag>::T T;
  constexpr int P = 4 * KS, ROWS = 64 / P;   // pieces of 16 bytes a row; rows a transfer
  __shared__ __attribute__((aligned(16))) char smem[BM * P * 16];
  const MvBlockLinearArgs &p = q.a;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4;
  // (workgroups are dealt to the 8 XCDs in turn: each gets a run of rows, all outputs of 128 one behind the other)
  const int id = blockIdx.x, more = gridDim.x & 7, at = (id & 7) * (gridDim.x >> 3) + min(id & 7, more) + (id >> 3), m0 = at / q.all * BM, tile = at % q.all;
  int b = 0;
#pragma unroll
  for (int i = 1; i < MV_BLOCK_LINEAR_MAX; ++i)
    if (i < p.blocks && tile >= q.tiles[i]) b = i;
  const int n0 = p.first_output[b] + (tile - q.tiles[b]) * BN, n_end = p.first_output[b] + p.outputs[b], k0 = p.first_input[b];
#pragma unroll
  for (int i = 0; i < BM / ROWS / 4; ++i) {
    const int f = i * 4 + wave, row = f * ROWS + lane / P, piece = (lane % P) ^ (row & (P - 1));   // (an order that spreads the rows over the banks)
    const T *from = (const T *)p.x + (int64_t)min(m0 + row, p.rows - 1) * p.x_stride + k0 + piece * 8;
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)from, (__attribute__((address_space(3))) void *)(smem + f * 1024), 16, 0, 0);
  }
  const int wm = (wave & 1) * 64, wn = n0 + (wave >> 1) * 64;
  u32x4 w[4][KS];   // row r16 of tile j: output 32 (j >> 1) + 8 (r16 >> 2) + 4 (j & 1) + (r16 & 3)
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = min(wn + 32 * (j >> 1) + 8 * (r16 >> 2) + 4 * (j & 1) + (r16 & 3), n_end - 1);
    const T *row = (const T *)p.w + (int64_t)n * p.k + k0 + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) w[j][s] = *(const u32x4 *)(row + 32 * s);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    u32x4 x[KS];
    const int row = wm + 16 * i + r16;
#pragma unroll
    for (int s = 0; s < KS; ++s) x[s] = *(const u32x4 *)(smem + row * P * 16 + ((4 * s + g) ^ (row & (P - 1))) * 16);
    f32x4 acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = mfma16x16x32<Tag>(w[j][s], x[s], acc[j]);
    if (m0 + row >= p.rows) continue;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int n = wn + 32 * h + 8 * g;
      if (n >= n_end) continue;
      const u32x2 lo = pack_quad<Tag>(acc[2 * h]), hi = pack_quad<Tag>(acc[2 * h + 1]);
      *(u32x4 *)((T *)p.out + (int64_t)(m0 + row) * p.out_stride + n) = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
  }
}

}  // namespace

extern "C" int mv_block_linear(const MvBlockLinearArgs *a, int dtype, void *stream) {
  if (a && a->rows == 0) return MV_OK;
  if (!a || !a->x || !a->w || !a->out) return MV_E_NULLPTR;
  if (dtype != MV_BF16 && dtype != MV_F16) return MV_E_DTYPE;
  if (a->rows < 0 || a->blocks < 1 || a->blocks > MV_BLOCK_LINEAR_MAX || (a->inputs != 64 && a->inputs != 128) || (a->k & 7)) return MV_E_SHAPE;
  BlockLinear q{*a, {}, 0};
  int64_t tiles = 0;
  for (int b = 0; b < a->blocks; ++b) {
    if (a->outputs[b] <= 0 || (a->outputs[b] & 7) || (a->first_output[b] & 7) || a->first_output[b] < 0 || a->first_input[b] < 0 || (a->first_input[b] & 7) ||
        a->first_input[b] + a->inputs > a->k || a->first_input[b] + a->inputs > a->x_stride || (int64_t)a->first_output[b] + a->outputs[b] > a->out_stride)
      return MV_E_SHAPE;
    q.tiles[b] = (int)tiles;
    tiles += (a->outputs[b] + BN - 1) / BN;
  }
  q.all = (int)tiles;
  const int64_t all = tiles * (((int64_t)a->rows + BM - 1) / BM);
  if (all > 0x7fffffff) return MV_E_SHAPE;
  if (!mv_aligned16(a->x) || !mv_aligned16(a->w) || !mv_aligned16(a->out) || (a->x_stride & 7) || (a->out_stride & 7)) return MV_E_ALIGN;
  const dim3 grid((unsigned)all);
#define MV_BL(Tag_, KS_) hipLaunchKernelGGL((block_linear_kernel<Tag_, KS_>), grid, dim3(256), 0, (hipStream_t)stream, q)
  if (dtype == MV_BF16) {
    if (a->inputs == 64) MV_BL(bf16_tag, 2);
    else MV_BL(bf16_tag, 4);
  } else {
    if (a->inputs == 64) MV_BL(f16_tag, 2);
    else MV_BL(f16_tag, 4);
  }
#undef MV_BL
  MV_LAUNCH_CHECK();
  return MV_OK;
}
