// K21 — fp32 projections on the 16-bit matrix cores: out = max(x W^T + bias, 0) + residual, operands in parts.
//
// A number of fp32 from 2^-109 on is the sum of three of bf16 (24 bits of significand), and a product is the six of its parts' products that matter: what is
// left out is 2^-24 of it at the most.  Smaller numbers that are not (bf16 ends at 2^-133) go as their own 32 bits beside a NaN (parts.h), and fragments with results that
// are not finite are made once more from the numbers by fp32 matrix instructions: 6470 rows of 768 -> 3072, parts and product, us: 180 (library 301), one such number in
// x, or a NaN, 303, an output all of whose weights are 218, an input whose weights all are 1106.  A product of parts is exact and sums are fp32, those of the first parts apart from the rest, so that the rest's
// roundings do not count; a matrix instruction adds 32 products at once.  Distance from 64 bits, relative, unit normal inputs: 768 inputs 1.6e-7 (library: 5.0e-7,
// few rows 2.5e-7), 3072 that are not negative 2.7e-7 (6.9e-7, 3.5e-7).  Six bf16 products take less time than one of fp32 (a sixteenth of the rate).
//
// mv_split_f32 brings operands into parts, in the order in which the products read them (weights too, for each call: nothing is kept that could be out
// of date); a LayerNorm in front of x rides in it, and a projection whose result only feeds another one writes parts itself.
// Parts made on the way into LDS instead, again for each tile: 768 -> 3072, 6470 rows 174 us where this takes 149 + 14.
//
// Bound by power: at 128 x 128 outputs a workgroup, two a CU, the matrix cores are busy 85 % of the time, at 1.6 GHz of 2.4 (operands of zeros: 2.3).  Hence
// 16 x 16 x 32 instructions: in registers alone they reach 2010 TFLOP/s at 2.0 GHz where 32 x 32 x 16 reach 1770 at 1.76 (of zeros both 2450), here
// 168 us -> 149.  LDS holds five stages of one part of 32 inputs; transfers are asked for between products (all at the start of a stage: 183 us, as waves
// stand still until theirs are taken).  Tiles of 64 x 64, six a CU with three stages each (parts written: five, four), where there are not enough of the larger ones
// (four with five stages: 768 inputs to 768 outputs, 6470 rows 48 us where this takes 44, 3072 to 768 174, 158; tiles of 64 x 128, three a CU 47, 162).
// us, library / this, with parts made of both operands: 6470 rows of 768 -> 2304 203 / 128, 768 -> 768 88 / 54, 768 -> 3072 280 / 166, 3072 -> 768 233 / 184;
// 1300 rows of 768 -> 3072 56 / 47; 8000 of 2048 -> 12288 2772 / 1715.
#include <algorithm>

#include "parts.h"

namespace {

// Parts lie as the products read them: [16 rows][32 inputs][part][quarter of the inputs, row][8]
__device__ __forceinline__ int64_t part_place(int64_t row, int piece, int k) { return ((row >> 4) * (k >> 5) + (piece >> 2)) * 192 + (piece & 3) * 16 + (row & 15); }

constexpr int kSpan = 1024;   // inputs of 16 rows for a workgroup
struct Split {
  MvSplitF32Args a;
  int first[MV_SPLIT_F32_MAX];   // workgroup of each matrix
};

__global__ void __launch_bounds__(256) split_f32_kernel(Split q) {
  const MvSplitF32Args &p = q.a;
  int m = 0;
#pragma unroll
  for (int i = 1; i < MV_SPLIT_F32_MAX; ++i)
    if (i < p.count && (int)blockIdx.x >= q.first[i]) m = i;
  const int k = p.k[m], rows = p.rows[m], spans = (k + kSpan - 1) / kSpan, at = blockIdx.x - q.first[m], row0 = at / spans * 16, k0 = at % spans * kSpan;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // A wave takes 16 rows x 32 inputs at a time, four lanes a row, and holds all that it takes of the span; rows behind the end repeat the last one.
  constexpr int TAKES = kSpan / 128;
  const float *src = (const float *)p.src[m] + (int64_t)min(row0 + (lane >> 2), rows - 1) * p.stride[m] + (lane & 3) * 8;
  f32x4 v[TAKES][2];
  auto load = [&](int from) {   // takes of the span at `from` that are there
    const int takes = (min(kSpan, k - from) / 32 - wave + 3) / 4;
#pragma unroll
    for (int t = 0; t < TAKES; ++t)
      if (t < takes) {
        const float *at = src + from + (t * 4 + wave) * 32;
        v[t][0] = *(const f32x4 *)at, v[t][1] = *(const f32x4 *)(at + 4);
      }
    return takes;
  };
  const bool norm = m == 0 && p.norm_w;
  float mean = 0.f, scale = 1.f;
  int takes;
  if (norm) {   // a row's sums, over its four lanes and the waves: of the numbers, of the squares of what they are off the mean
    __shared__ float sums[2][4][16];
    auto sum_of = [&](float x, int which) {
      x = lanes_sum<4>(x);
      if ((lane & 3) == 0) sums[which][wave][lane >> 2] = x;
      __syncthreads();
      return (sums[which][0][lane >> 2] + sums[which][1][lane >> 2]) + (sums[which][2][lane >> 2] + sums[which][3][lane >> 2]);
    };
    float sum = 0.f, square = 0.f;
    for (int i = 1; i <= spans; ++i) {   // (the own span last, which stays)
      takes = load((k0 / kSpan + i) % spans * kSpan);
#pragma unroll
      for (int t = 0; t < TAKES; ++t)
        if (t < takes) {
          const f32x4 both = v[t][0] + v[t][1];
          sum += (both[0] + both[1]) + (both[2] + both[3]);
        }
    }
    mean = sum_of(sum, 0) / (float)k;
    for (int i = 0; i < spans; ++i) {
      if (i) takes = load((k0 / kSpan + i) % spans * kSpan);
#pragma unroll
      for (int t = 0; t < TAKES; ++t)
        if (t < takes) {
          const f32x4 a = v[t][0] - mean, b = v[t][1] - mean, both = a * a + b * b;
          square += (both[0] + both[1]) + (both[2] + both[3]);
        }
    }
    scale = 1.f / sqrtf(sum_of(square, 1) / (float)k + p.eps);
  }
  if (!norm || spans > 1) takes = load(k0);
#pragma unroll
  for (int t = 0; t < TAKES; ++t)
    if (t < takes) {
      const int i = k0 + (t * 4 + wave) * 32 + (lane & 3) * 8;
      if (norm)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 w = *(const f32x4 *)((const float *)p.norm_w + i + 4 * h), b = p.norm_b ? *(const f32x4 *)((const float *)p.norm_b + i + 4 * h) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int n = 0; n < 4; ++n) v[t][h][n] = fmaf((v[t][h][n] - mean) * scale, w[n], b[n]);
        }
      float f[8] = {v[t][0][0], v[t][0][1], v[t][0][2], v[t][0][3], v[t][1][0], v[t][1][1], v[t][1][2], v[t][1][3]};
      u32x4 part[3];
      split3<true>(f, part);
      u32x4 *to = (u32x4 *)p.dst[m] + part_place(row0 + (lane >> 2), i >> 3, k);
#pragma unroll
      for (int s = 0; s < 3; ++s) to[64 * s] = part[s];
    }
}

// 32 XT rows x 32 WT outputs of 2 x 2 waves; workgroups of a CU; stages in LDS
template <int XT, int WT, int BESIDE, int SLOTS, bool PARTS>
__global__ void __launch_bounds__(256, BESIDE) linear_f32_kernel(MvLinearF32Args p, int mt, int nt) {
  constexpr int PIECES = 2 * (XT + WT), PER = PIECES / 4, STAGE = PIECES * 1024, kSlots = SLOTS;   // PIECES: fragments of 1 KiB; PER: of a wave
  static_assert(PIECES % 4 == 0 && PER <= WT);
  extern __shared__ __attribute__((aligned(16))) char smem[];   // stages of one part of 32 inputs: rows [2 XT] | weights [2 WT]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4, wm = wave & 1, wn = wave >> 1;
  const int id = blockIdx.x, more = gridDim.x & 7, at = (id & 7) * (gridDim.x >> 3) + min(id & 7, more) + (id >> 3);
  const int group = at / (8 * nt), in = at - group * 8 * nt, high = min(8, mt - group * 8);
  const int mi = group * 8 + in % high, ni = in / high, stages = p.k / 32 * 3;
  const int last_x = (p.rows - 1) >> 4, last_w = (p.n - 1) >> 4;
  const char *src[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int t = i * 4 + wave;
    const int64_t tile = t < 2 * XT ? min(mi * 2 * XT + t, last_x) : min(ni * 2 * WT + t - 2 * XT, last_w);
    src[i] = (const char *)(t < 2 * XT ? p.x : p.w) + tile * stages * 1024 + lane * 16;
  }
  auto fetch = [&](int i, int slot) __attribute__((always_inline)) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src[i],
                                     (__attribute__((address_space(3))) void *)(smem + slot * STAGE + (i * 4 + wave) * 1024), 16, 0, 0);
    src[i] += 1024;
  };
  f32x4 acc[WT][XT] = {}, low[WT][XT] = {};   // the products of the first parts; the others
  const uint32_t xa = lds_address(smem) + lane * 16 + wm * XT * 1024, wa = lds_address(smem) + lane * 16 + (2 * XT + wn * WT) * 1024;
  u32x4 x[2][XT], w[2][WT];   // the first part; the part of the stage
  for (int t = 0; t < min(kSlots - 1, stages); ++t)
#pragma unroll
    for (int i = 0; i < PER; ++i) fetch(i, t);
  int slot = 0;
  auto stage = [&](auto P, int s) __attribute__((always_inline)) {
    constexpr int part = decltype(P)::value, at = part ? 1 : 0;
    // stage s is there, and every wave is past stage s - 1, whose place the one that is asked for now takes
    if (s + kSlots - 2 < stages) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER * (kSlots - 2)) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    const bool ahead = s + kSlots - 1 < stages;
    const int free = slot == 0 ? kSlots - 1 : slot - 1;
    const uint32_t xs = xa + slot * STAGE, ws = wa + slot * STAGE;
    slot = slot == kSlots - 1 ? 0 : slot + 1;
    static_for<XT>([&](auto I) { lds_read128<decltype(I)::value * 1024>(x[at][decltype(I)::value], xs); });
    static_for<WT>([&](auto I) { lds_read128<decltype(I)::value * 1024>(w[at][decltype(I)::value], ws); });
    auto product = [&](f32x4 (&to)[WT][XT], const u32x4 (&w)[WT], const u32x4 (&x)[XT], int first, int pieces) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < WT; ++j) {
        __builtin_amdgcn_sched_barrier(0);
        if (ahead && j < pieces) fetch(first + j, free);
#pragma unroll
        for (int i = 0; i < XT; ++i) to[j][i] = mfma16x16x32<bf16_tag>(w[j], x[i], to[j][i]);
      }
    };
    static_for<XT>([&](auto I) { lds_wait<WT>(x[at][decltype(I)::value]); });
    if constexpr (part) product(low, w[0], x[1], 0, PER);
    static_for<WT>([&](auto I) { lds_wait<0>(w[at][decltype(I)::value]); });
    if constexpr (part == 0) product(acc, w[0], x[0], 0, PER);
    if constexpr (part == 1) product(low, w[1], x[0], 0, 0), product(low, w[1], x[1], 0, 0);
    if constexpr (part == 2) product(low, w[1], x[0], 0, 0);
  };
  for (int s = 0; s < stages; s += 3) static_for<3>([&](auto P) { stage(P, s + decltype(P)::value); });
  lds_barrier();
  constexpr int COLS = WT * 16, ROW = COLS * 4 + 16;   // a wave's outputs; bytes of a row of them in LDS
  char *const tile = smem + wave * (32 * ROW);
  const int first = (ni * 2 + wn) * COLS;
  // A fragment of 16 rows x 16 outputs some of whose products are not finite, once more by fp32 matrix instructions from the numbers themselves
  auto again = [&](int i, int j) {
    const char *xr = (const char *)p.x + (int64_t)min(mi * 2 * XT + wm * XT + i, last_x) * stages * 1024 + lane * 16;
    const char *wr = (const char *)p.w + (int64_t)min(ni * 2 * WT + wn * WT + j, last_w) * stages * 1024 + lane * 16;
    f32x4 sum[2] = {};
    for (int s = 0; s < stages; s += 3, xr += 3072, wr += 3072) {
      u32x4 xp[3], wp[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) xp[q] = *(const u32x4 *)(xr + q * 1024), wp[q] = *(const u32x4 *)(wr + q * 1024);
      float xn[8], wn[8];
      joined8(xp, xn), joined8(wp, wn);
#pragma unroll
      for (int q = 0; q < 8; ++q) sum[q & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(wn[q], xn[q], sum[q & 1], 0, 0, 0);
    }
    return sum[0] + sum[1];
  };
  auto finish = [&](f32x4 v, int n) __attribute__((always_inline)) {
    if (p.bias) v += *(const f32x4 *)((const float *)p.bias + n);
    if (p.relu) {
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = v[q] < 0.f ? 0.f : v[q];   // (NaN stays)
    }
    return v;
  };
#pragma unroll
  for (int i = 0; i < XT; i += 2) {   // 32 rows at a time
    uint32_t odd = 0;   // fragments that have a number that is not finite
#pragma unroll
    for (int j = 0; j < WT; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4 v = acc[j][i + h] + low[j][i + h];
        *(f32x4 *)(tile + (h * 16 + r16) * ROW + j * 64 + g * 16) = v;
        uint32_t largest = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) largest = max(largest, f2u(v[q]) & 0x7fffffffu);
        if (__any(largest >= 0x7f800000u)) odd |= 1u << (2 * j + h);
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    for (; odd; odd &= odd - 1) {
      const int at = __builtin_ctz(odd), h = at & 1, j = at >> 1;
      const f32x4 sum = again(i + h, j);
      f32x4 *const of = (f32x4 *)(tile + (h * 16 + r16) * ROW + j * 64 + g * 16);
      f32x4 v = *of;
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = fabsf(v[q]) < INFINITY ? v[q] : sum[q];
      *of = v;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    const int row0 = (mi * 2 + wm) * XT * 16 + i * 16;
    if constexpr (PARTS) {
#pragma unroll
      for (int r = 0; r < COLS / 16; ++r) {   // 16 rows x 32 outputs
        const int in_tile = r / (COLS / 32) * 16 + r16, row = row0 + in_tile, at = r % (COLS / 32) * 32 + g * 8, n = first + at;
        const float *from = (const float *)(tile + in_tile * ROW) + at;
        if (row - r16 >= p.rows || n >= p.n) continue;   // (rows behind the end, up to a whole tile, are written too: nobody's results depend on them)
        f32x4 a = finish(*(const f32x4 *)from, n), b = finish(*(const f32x4 *)(from + 4), n + 4);
        float f[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
        u32x4 part[3];
        split3<true>(f, part);
        u32x4 *to = (u32x4 *)p.out + part_place(row, n >> 3, p.n);
#pragma unroll
        for (int s = 0; s < 3; ++s) to[64 * s] = part[s];
      }
    } else {
      constexpr int LINE = COLS / 4;
      const int n = first + lane % LINE * 4;
#pragma unroll
      for (int r = 0; r < 32 * LINE / 64; ++r) {
        const int in_tile = r * (64 / LINE) + lane / LINE, row = row0 + in_tile;
        if (row >= p.rows || n >= p.n) continue;
        f32x4 v = finish(*(const f32x4 *)(tile + in_tile * ROW + lane % LINE * 16), n);
        if (p.residual) v += *(const f32x4 *)((const float *)p.residual + (int64_t)row * p.residual_stride + n);
        *(f32x4 *)((float *)p.out + (int64_t)row * p.out_stride + n) = v;
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
}

template <int XT, int WT, int BESIDE, int SLOTS, bool PARTS>
int launch(const MvLinearF32Args &p, hipStream_t st) {
  const int64_t mt = ((int64_t)p.rows + 32 * XT - 1) / (32 * XT), nt = ((int64_t)p.n + 32 * WT - 1) / (32 * WT);
  if (mt * nt > 0x7fffffff) return MV_E_SHAPE;
  if (int rc = mv_allow_lds<linear_f32_kernel<XT, WT, BESIDE, SLOTS, PARTS>>()) return rc;
  constexpr int lds = SLOTS * (XT + WT) * 2048;
  hipLaunchKernelGGL((linear_f32_kernel<XT, WT, BESIDE, SLOTS, PARTS>), dim3((unsigned)(mt * nt)), dim3(256), lds, st, p, (int)mt, (int)nt);
  MV_LAUNCH_CHECK();
  return MV_OK;
}

}  // namespace

extern "C" size_t mv_split_f32_bytes(int rows, int k) { return rows < 1 || k < 1 || (k & 31) ? 0 : (size_t)((rows + 15) / 16) * (k / 32) * 3072; }

extern "C" int mv_split_f32(const MvSplitF32Args *a, void *stream) {
  if (!a) return MV_E_NULLPTR;
  if (a->count < 1 || a->count > MV_SPLIT_F32_MAX) return MV_E_SHAPE;
  Split q{*a, {}};
  int64_t all = 0;
  for (int i = 0; i < a->count; ++i) {
    if (!a->src[i] || !a->dst[i]) return MV_E_NULLPTR;
    if (a->rows[i] < 1 || a->k[i] < 32 || (a->k[i] & 31) || a->stride[i] < a->k[i]) return MV_E_SHAPE;
    if (!mv_aligned16(a->src[i]) || !mv_aligned16(a->dst[i]) || (a->stride[i] & 3)) return MV_E_ALIGN;
    q.first[i] = (int)all;
    all += ((int64_t)a->rows[i] + 15) / 16 * ((a->k[i] + kSpan - 1) / kSpan);
    if (all > 0x7fffffff) return MV_E_SHAPE;
  }
  if (!mv_aligned16(a->norm_w) || !mv_aligned16(a->norm_b)) return MV_E_ALIGN;
  hipLaunchKernelGGL(split_f32_kernel, dim3((unsigned)all), dim3(256), 0, (hipStream_t)stream, q);
  MV_LAUNCH_CHECK();
  return MV_OK;
}

extern "C" int mv_linear_f32(const MvLinearF32Args *a, void *stream) {
  if (a && a->rows == 0) return MV_OK;
  if (!a || !a->x || !a->w || !a->out) return MV_E_NULLPTR;
  if (a->tile < 0 || a->tile > 2) return MV_E_RANGE;
  if (a->rows < 0 || a->n <= 0 || a->k <= 0 || (a->n & 3) || (a->k & 31) || (a->parts_out && (a->n & 31)) || (!a->parts_out && a->out_stride < a->n) ||
      (a->residual && (a->parts_out || a->residual_stride < a->n)))
    return MV_E_SHAPE;
  if (!mv_aligned16(a->x) || !mv_aligned16(a->w) || !mv_aligned16(a->out) || !mv_aligned16(a->bias) || !mv_aligned16(a->residual) ||
      (!a->parts_out && (a->out_stride & 3)) || (a->residual && (a->residual_stride & 3)))
    return MV_E_ALIGN;
  hipStream_t st = (hipStream_t)stream;
  // 512 tiles of 128 x 128 run at a time: those where their last round is well filled, or there are many.  us, 64 x 64 / 128 x 128, by tiles of 128 x 128:
  // 384 52 / 60, 416 of 2048 inputs 144 / 147 and 146 / 142, 468 65 / 62, 504 66 / 64, 594 80 / 89, 624 82 / 90, 720 95 / 96, 792 103 / 113, 832 265 / 277, 918 118 / 116,
  // 960 120 / 119, 1008 324 / 300, 1056 343 / 339 and 321 / 337, 1134 147 / 148, 1224 155 / 151, 1280 400 / 363, 1422 180 / 176, 2016 638 / 571
  const int64_t wide = (((int64_t)a->rows + 127) / 128) * (((int64_t)a->n + 127) / 128);
  const bool large = a->tile == 1 || (a->tile == 0 && (wide >= 1150 || wide * 100 >= (wide + 511) / 512 * 512 * 85));
  if (large) return a->parts_out ? launch<4, 4, 2, 5, true>(*a, st) : launch<4, 4, 2, 5, false>(*a, st);
  return a->parts_out ? launch<2, 2, 5, 4, true>(*a, st) : launch<2, 2, 6, 3, false>(*a, st);
}
