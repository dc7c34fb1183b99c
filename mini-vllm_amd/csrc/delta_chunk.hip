// K16 — gated delta rule of prompts in chunks of 64 tokens on the matrix cores (16-bit operands, fp32 state).
//
// With r_i the running sum of the log decays in a chunk (per key channel), k and q scaled to their lengths, S the state ahead of the
// chunk and all vectors rows, the recurrence unrolls to
//     u_i = beta_i (v_i - (e^{r_i} k_i) S - sum_{j < i} A_ij u_j),    A_ij = sum_c k_ic k_jc e^{r_ic - r_jc}
//     o_i = (e^{r_i} q_i) S + sum_{j <= i} B_ij u_j,                  B_ij = sum_c q_ic k_jc e^{r_ic - r_jc}
//     S  <- e^{r_last} S + sum_j (e^{r_last - r_j} k_j)^T u_j
// The u of a chunk solve a unit lower triangular system: with T = (1 + A)^-1 diag(beta), U = U0 - W S, U0 = T v, W = T e^r k.
// Two launches:
//   prepare: everything that does not need S, one workgroup per (chunk, head): A, B, T, U0, W, the scaled operands;
//   walk:    chunks one behind the other, one workgroup per (sequence, head, columns): four products with S and U.
// What is fp32 by nature enters a product as the sum of two bf16 numbers (three MFMAs: high x high, high x rest, rest x high), about
// 16 bits of mantissa.  The operands lie in the workspace as MFMA fragments (64 lanes x 16 bytes), which the walk fetches by LDS-DMA.
//
// One decay per head needs less (delta_scalar.hip, bf16).
//
// Exponentials never overflow: A and B are computed by blocks of 16 x 16 tokens with the sums taken relative to r at the end of the
// block in front of the rows' (both factors at most 1), or in the middle of a diagonal block; where a block decays by more than
// 2^kRange a diagonal block is summed pair by pair instead.
#include <algorithm>
#include <cmath>

#include "delta_chunk.h"

namespace {

typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

constexpr float kRange = 60.f;     // log2
constexpr int kPrepareWaves = 8;

// sizes of a (chunk, head) in the workspace, in fragments of 1 KiB: [W | Q: 4 token tiles][NK][high, rest] | U0: 4 per 16 columns |
// K: [2 NK state tiles][2][high, rest] | B: [4 token tiles][2][high, rest] | decay of the whole chunk
struct Layout {
  int u0, k, b, tail, total;
  __host__ __device__ constexpr Layout(int nk, int p) : u0(16 * nk), k(16 * nk + p / 4), b(24 * nk + p / 4), tail(24 * nk + p / 4 + 16), total(24 * nk + p / 4 + 17) {}
};

// Workgroup = 8 waves of a (chunk, head).  Bound by its vector arithmetic (some 15 000 instructions of a wave, a tenth of them exponentials) and by the latency
// of its phases: everything is asked for from memory at the start, blocks of one row of A and B share that row's factors, K is made beside the
// solution, and the solution is split into operands once.  3 sequences of 4011 tokens and less, 8 heads of 128 x 128 (1256 workgroups, two a CU):
// 105 us with every block's factors, all of K and W by four waves, and operands of T by each item -> 83.
// CONV (q.raw: projected channels, all of this head's alone): convolution and silu ahead of it (conv_chunk), k and q into their place in LDS, v by way of the decays' place
// into registers.  Nobody else reads the convolved channels, so they leave the CU no more: a launch and 77 MB less.  The sequences above: 32 + 85 us as two launches, the
// layer 250 -> 232.
template <typename Tag, int NK, bool CONV>
__global__ void __launch_bounds__(kPrepareWaves * 64, NK < 5 ? 4 : 2) delta_prepare_kernel(DeltaPrep q) {
  typedef typename elem<Tag>::T T;
  constexpr int N = NK * 32, W = kPrepareWaves, RS = N + 4, KS = N + 8;   // LDS row strides: fp32, 16-bit
  static_assert(W == 8, "the blocks are dealt to eight waves");
  const MvDeltaArgs &p = q.a;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float *rs = (float *)smem;                              // [L][RS] running log2 decays
  T *ks = (T *)(smem + L * RS * 4), *qs = ks + L * KS;    // [L][KS]; later (from qs on) -A, then T, then its operands
  float *ts = (float *)qs;                                // [L][TS]
  constexpr int QB = L * KS * 2 > L * TS * 4 ? L * KS * 2 : L * TS * 4;
  float *fk = (float *)((char *)qs + QB), *fq = fk + L, *bt = fq + L, *part_sums = bt + L;   // [W][64]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
  const int head = blockIdx.y;
  const int seq = chunk_sequence(p, blockIdx.x);
  const int q0 = p.cu_q[seq], len = p.cu_q[seq + 1] - q0, t0 = ((int)blockIdx.x - q0 / L - seq) * L;
  if (t0 >= len) return;
  const int nt = min(L, len - t0), grp = head / (p.heads / p.groups);
  const Layout lay(NK, p.p);
  char *ws = q.ws + ((int64_t)blockIdx.x * p.heads + head) * lay.total * 1024;
  const T *x = (const T *)p.x + (int64_t)(q0 + t0) * p.x_stride;

  // ---- everything that comes from memory: k and q, eight threads a token; the decays; v of this wave's (first) 16 columns
  constexpr int KQ = (N + 63) / 64, AP = (L * N / 8 + W * 64 - 1) / (W * 64);   // pieces of 8 channels a thread
  const int tt = tid >> 3, part = tid & 7, columns = p.p / 16;
  u32x4 kraw[KQ], qraw[KQ], araw[AP], braw[AP];
  if constexpr (!CONV) {
    const T *row = x + (int64_t)min(tt, nt - 1) * p.x_stride + grp * N;
#pragma unroll
    for (int i = 0; i < KQ; ++i) {
      const int c = min(part * 8 + 64 * i, N - 8);
      kraw[i] = *(const u32x4 *)(row + p.k_off + c), qraw[i] = *(const u32x4 *)(row + p.q_off + c);
    }
  }
  const T *a = (const T *)p.a + (int64_t)(q0 + t0) * p.a_stride, *bias = (const T *)p.dt_bias;
  const T *of_beta = (const T *)p.beta + (int64_t)(q0 + t0 + min(tt, nt - 1)) * p.beta_stride + head;
  const float beta = elem<Tag>::ld(*of_beta), log_rate = elem<Tag>::ld(((const T *)p.a_log)[head]);
  float a_head = 0.f, b_head = 0.f;
  if (p.channel_decay) {
#pragma unroll
    for (int i = 0; i < AP; ++i) {
      const int at = min(tid + i * W * 64, L * N / 8 - 1), t = at / (N / 8), c = (at - t * (N / 8)) * 8;
      araw[i] = *(const u32x4 *)(a + (int64_t)min(t, nt - 1) * p.a_stride + head * N + c);
      braw[i] = *(const u32x4 *)(bias + head * N + c);
    }
  } else {
    a_head = elem<Tag>::ld(a[(int64_t)min(tt, nt - 1) * p.a_stride + head]), b_head = elem<Tag>::ld(bias[head]);
  }
  T vraw[16];
  auto load_values = [&](int ct) __attribute__((always_inline)) {
    const T *v = x + head * p.p + ct * 16 + r16;
#pragma unroll
    for (int e = 0; e < 16; ++e) vraw[e] = v[(int64_t)min(16 * (e >> 2) + 4 * g + (e & 3), nt - 1) * p.x_stride];
  };
  if constexpr (CONV) {
    T *vs = (T *)smem;   // [L][VS], where the decays' sums come later
    const int VS = p.p + 8;
    conv_chunk<Tag, N, W * 64, true>(q, seq, q0, len, t0, nt, head, head * p.p, p.p, tid, [&](int which, int row, int at, int, u32x2 done) {
      *(u32x2 *)(which == 0 ? ks + row * KS + at : which == 1 ? qs + row * KS + at : vs + row * VS + at) = done;
    });
    __syncthreads();
#pragma unroll
    for (int i = 0; i < KQ; ++i) {
      const int c = min(part * 8 + 64 * i, N - 8);
      kraw[i] = *(const u32x4 *)(ks + tt * KS + c), qraw[i] = *(const u32x4 *)(qs + tt * KS + c);
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) vraw[e] = vs[(16 * (e >> 2) + 4 * g + (e & 3)) * VS + min(wave, columns - 1) * 16 + r16];
    __syncthreads();
  } else {
    load_values(min(wave, columns - 1));
  }

  // ---- k, q (tokens behind the end: zeros) and their lengths
  {
    float sk = 0.f, sq = 0.f;
#pragma unroll
    for (int i = 0; i < KQ; ++i) {
      const int c = part * 8 + 64 * i;
      if (N % 64 && c >= N) continue;
      if (tt >= nt) kraw[i] = qraw[i] = u32x4{0u, 0u, 0u, 0u};
      float fa[8], fb[8];
      unpack8<Tag>(kraw[i], fa);
      unpack8<Tag>(qraw[i], fb);
#pragma unroll
      for (int j = 0; j < 8; ++j) sk = fmaf(fa[j], fa[j], sk), sq = fmaf(fb[j], fb[j], sq);
      if constexpr (!CONV) {
        *(u32x4 *)(ks + tt * KS + c) = kraw[i];
        *(u32x4 *)(qs + tt * KS + c) = qraw[i];
      }
    }
#pragma unroll
    for (int o = 1; o <= 4; o <<= 1) sk += __shfl_xor(sk, o, 64), sq += __shfl_xor(sq, o, 64);
    if (part == 0) {
      fk[tt] = 1.f / sqrtf(sk + p.unit_eps), fq[tt] = p.q_scale / sqrtf(sq + p.unit_eps);
      bt[tt] = tt < nt ? sigmoid_f32(beta) : 0.f;
    }
  }
  // ---- log2 decays, summed over the tokens
  {
    const float rate = -expf(log_rate) * 1.4426950408889634f;
    if (p.channel_decay) {
#pragma unroll
      for (int i = 0; i < AP; ++i) {
        const int at = tid + i * W * 64, t = at / (N / 8), c = (at - t * (N / 8)) * 8;
        if (L * N / 8 % (W * 64) && at >= L * N / 8) continue;
        float f[8], b[8];
        unpack8<Tag>(araw[i], f);
        unpack8<Tag>(braw[i], b);
#pragma unroll
        for (int j = 0; j < 8; ++j) f[j] = t < nt ? rate * softplus_fast(f[j] + b[j]) : 0.f;
        f32x4 *dst = (f32x4 *)(rs + t * RS + c);
        dst[0] = f32x4{f[0], f[1], f[2], f[3]}, dst[1] = f32x4{f[4], f[5], f[6], f[7]};
      }
    } else {
      const float v = tt < nt ? rate * softplus_fast(a_head + b_head) : 0.f;
      for (int c = part; c < N; c += 8) rs[tt * RS + c] = v;
    }
    __syncthreads();
    // a thread TW of a channel's tokens (the threads of a wave: adjacent channels); then the sums ahead are added
    constexpr int TW = L / W;
    for (int c0 = 0; c0 < N; c0 += 64) {
      const int c = c0 + lane;
      float v[TW], sum = 0.f;
      if (c < N) {
#pragma unroll
        for (int t = 0; t < TW; ++t) v[t] = rs[(TW * wave + t) * RS + c];
#pragma unroll
        for (int t = 0; t < TW; ++t) sum += v[t], v[t] = sum;
        part_sums[wave * 64 + lane] = sum;
      }
      __syncthreads();
      if (c < N) {
        float ahead = 0.f;
#pragma unroll
        for (int w = 0; w < W - 1; ++w) ahead += w < wave ? part_sums[w * 64 + lane] : 0.f;
#pragma unroll
        for (int t = 0; t < TW; ++t) rs[(TW * wave + t) * RS + c] = ahead + v[t];
      }
      if (c0 + 64 < N) __syncthreads();
    }
  }
  __syncthreads();

  // ---- A and B by blocks of 16 x 16 tokens (rows I, columns J <= I); a lane gets row r16, columns 4 g ..  A wave has one diagonal block or one or two
  // others of a row, which share the row's factors: 3: 0 1 | 2: 0 1 | 3: 2 | 1: 0 | the diagonal
  const int I = wave >= 4 ? 7 - wave : wave == 3 ? 1 : wave == 1 ? 2 : 3, J0 = wave >= 4 ? I : wave == 2 ? 2 : 0, blocks = wave < 2 ? 2 : 1;
  f32x4 blkA[2], blkB[2];
  {
    const bool diagonal = wave >= 4;
    const int ref = diagonal ? 16 * I + 7 : 16 * I - 1;
    const float *ri = rs + (16 * I + r16) * RS + 8 * g, *rr = rs + ref * RS + 8 * g;
    const T *ki = ks + (16 * I + r16) * KS + 8 * g, *qi = qs + (16 * I + r16) * KS + 8 * g;
#pragma unroll
    for (int m = 0; m < 2; ++m) blkA[m] = blkB[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    bool fits = true;   // (the sums fall, so the ends of a diagonal block decide)
    if (diagonal)
      for (int c = lane; c < N; c += 64)
        fits = fits && rs[16 * I * RS + c] - rs[ref * RS + c] <= kRange && rs[ref * RS + c] - rs[(16 * I + 15) * RS + c] <= kRange;
#pragma unroll
    for (int s = 0; s < NK; ++s) {
      float fi[8], fp[8], rc[8];
      unpack8<Tag>(*(const u32x4 *)(ki + 32 * s), fi);
      unpack8<Tag>(*(const u32x4 *)(qi + 32 * s), fp);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4 ra = *(const f32x4 *)(ri + 32 * s + 4 * h), c = *(const f32x4 *)(rr + 32 * s + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float el = __builtin_amdgcn_exp2f(ra[e] - c[e]);
          fi[4 * h + e] *= el, fp[4 * h + e] *= el, rc[4 * h + e] = c[e];
        }
      }
      u32x4 ih, il, ph, pl;
      split8(fi, ih, il);
      split8(fp, ph, pl);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        if (m >= blocks) continue;
        const int j = 16 * (J0 + m) + r16;
        const float *rj = rs + j * RS + 8 * g + 32 * s;
        float fj[8];
        unpack8<Tag>(*(const u32x4 *)(ks + j * KS + 8 * g + 32 * s), fj);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 rb = *(const f32x4 *)(rj + 4 * h);
#pragma unroll
          for (int e = 0; e < 4; ++e) fj[4 * h + e] *= __builtin_amdgcn_exp2f(rc[4 * h + e] - rb[e]);
        }
        u32x4 jh, jl;
        split8(fj, jh, jl);
        blkA[m] = mfma3(jh, jl, ih, il, blkA[m]);
        blkB[m] = mfma3(jh, jl, ph, pl, blkB[m]);
      }
    }
    const int i = 16 * I + r16;
    if (diagonal && !__all(fits)) {
      const int j0 = 16 * I + 4 * g;
      for (int e = 0; e < 4; ++e) {
        float sa = 0.f, sb = 0.f;
        if (j0 + e <= i)
          for (int c = 0; c < N; ++c) {
            const float k = elem<Tag>::ld(ks[(j0 + e) * KS + c]) * __builtin_amdgcn_exp2f(rs[i * RS + c] - rs[(j0 + e) * RS + c]);
            sa = fmaf(elem<Tag>::ld(ks[i * KS + c]), k, sa);
            sb = fmaf(elem<Tag>::ld(qs[i * KS + c]), k, sb);
          }
        blkA[0][e] = sa, blkB[0][e] = sb;
      }
    }
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      if (m >= blocks) continue;
      const int J = J0 + m, j0 = 16 * J + 4 * g;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        blkA[m][e] = j0 + e < i ? -blkA[m][e] * (bt[i] * fk[i] * fk[j0 + e]) : 0.f;   // (the negative)
        blkB[m][e] = j0 + e <= i ? blkB[m][e] * (fq[i] * fk[j0 + e]) : 0.f;
      }
      // B as an operand whose k order is that of an accumulator pair: key 16 (e >> 2) + 4 g + (e & 3) of a step of 32
      u32x2 hi, lo;
      split4(blkB[m], hi, lo);
      u32x2 *dst = (u32x2 *)(ws + (lay.b + (I * 2 + (J >> 1)) * 2) * 1024 + lane * 16) + (J & 1);
      dst[0] = hi;
      dst[128] = lo;
      if (I == J && (I & 1) == 0) dst[1] = dst[129] = u32x2{0u, 0u};   // the columns behind, in the same step of 32
    }
  }

  // ---- e^r q by rows (the waves with one block)
  if (wave >= 2) {
    for (int f = wave - 2; f < 4 * NK; f += W - 2) {
      const int it = f / NK, s = f - it * NK, t = 16 * it + r16, c = 32 * s + 8 * g;
      float v[8];
      u32x4 hi, lo;
      unpack8<Tag>(*(const u32x4 *)(qs + t * KS + c), v);
      const float w = fq[t];
      const f32x4 r0 = *(const f32x4 *)(rs + t * RS + c), r1 = *(const f32x4 *)(rs + t * RS + c + 4);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] *= w * __builtin_amdgcn_exp2f(e < 4 ? r0[e & 3] : r1[e & 3]);
      split8(v, hi, lo);
      u32x4 *dst = (u32x4 *)(ws + (8 * NK + f * 2) * 1024) + lane;
      dst[0] = hi, dst[64] = lo;
    }
  }
  for (int c = tid; c < N; c += W * 64) ((float *)(ws + lay.tail * 1024))[c] = __builtin_amdgcn_exp2f(rs[(L - 1) * RS + c]);
  __syncthreads();   // q is done with
#pragma unroll
  for (int m = 0; m < 2; ++m)
    if (m < blocks) *(f32x4 *)(ts + (16 * I + r16) * TS + 16 * (J0 + m) + 4 * g) = blkA[m];
  __syncthreads();

  // k of a state tile (in the order of the walk's accumulators), scaled: tokens 32 s + 16 (e >> 2) + 4 g + (e & 3) of channel c; and its sums of decays
  auto columns_of = [&](int i, int s, int &c, float (&k)[8], float (&r)[8]) __attribute__((always_inline)) {
    c = (i >> 1) * 32 + (r16 >> 2) * 8 + (i & 1) * 4 + (r16 & 3);
    const T *from = ks + (32 * s + 4 * g + (r16 >> 2)) * KS + (i >> 1) * 32 + (r16 & 3) * 8 + (i & 1) * 4;
    u32x2 h[2];
#pragma unroll
    for (int e = 0; e < 2; ++e)
      h[e] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(from + 16 * e * KS)));
    unpack8<Tag>(u32x4{h[0][0], h[0][1], h[1][0], h[1][1]}, k);
    const f32x4 f0 = *(const f32x4 *)(fk + 32 * s + 4 * g), f1 = *(const f32x4 *)(fk + 32 * s + 16 + 4 * g);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      k[e] *= e < 4 ? f0[e & 3] : f1[e & 3];
      r[e] = rs[(32 * s + 16 * (e >> 2) + 4 * g + (e & 3)) * RS + c];
    }
  };
  // ---- K = e^(r_last - r) k by state rows, by the waves that have no part in the solution
  if (wave >= 4) {
    for (int f = wave - 4; f < 4 * NK; f += 4) {
      const int i = f >> 1, s = f & 1;
      int c;
      float k[8], r[8];
      columns_of(i, s, c, k, r);
      const float last = rs[(L - 1) * RS + c];
#pragma unroll
      for (int e = 0; e < 8; ++e) k[e] *= __builtin_amdgcn_exp2f(last - r[e]);
      u32x4 hi, lo;
      split8(k, hi, lo);
      u32x4 *dst = (u32x4 *)(ws + (lay.k + f * 2) * 1024) + lane;
      dst[0] = hi, dst[64] = lo;
    }
  }
  solve_chunk(ts, bt, wave, lane);
  {
    u32x4 hi, lo;
    if (wave < kTriangle) solution_operand(ts, wave, lane, hi, lo);
    __syncthreads();
    if (wave < kTriangle) {
      u32x4 *dst = (u32x4 *)qs + wave * 128 + lane;
      dst[0] = hi, dst[64] = lo;
    }
    __syncthreads();
  }
  const u32x4 *solution = (const u32x4 *)qs + lane;   // [kTriangle][high, rest][64]

  // ---- by 16 channels: -W = -T e^r k by tokens; by 16 columns of v: U0 = T v
  for (int i = wave; i < 2 * NK; i += W) {
    f32x4 acc[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) acc[it] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      int c;
      float k[8], r[8];
      columns_of(i, s, c, k, r);
#pragma unroll
      for (int e = 0; e < 8; ++e) k[e] *= __builtin_amdgcn_exp2f(r[e]);
      u32x4 hi, lo;
      split8(k, hi, lo);
#pragma unroll
      for (int it = 2 * s; it < 4; ++it) acc[it] = mfma3(hi, lo, solution[triangle(it, s) * 128], solution[triangle(it, s) * 128 + 64], acc[it]);
    }
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      u32x2 hi, lo;
      split4(-acc[it], hi, lo);
      u32x2 *dst = (u32x2 *)(ws + (it * NK + (i >> 1)) * 2 * 1024 + lane * 16) + (i & 1);
      dst[0] = hi, dst[128] = lo;
    }
  }
  for (int ct = wave; ct < columns; ct += W) {
    if (ct != wave) load_values(ct);
    f32x4 acc[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) acc[it] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      float f[8];
      u32x4 hi, lo;
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = elem<Tag>::ld(vraw[8 * s + e]);
      split8(f, hi, lo);
#pragma unroll
      for (int it = 2 * s; it < 4; ++it) {
        const u32x4 th = solution[triangle(it, s) * 128], tl = solution[triangle(it, s) * 128 + 64];
        acc[it] = mfma16x16x32<B16>(th, hi, acc[it]);
        acc[it] = mfma16x16x32<B16>(tl, hi, acc[it]);
        if constexpr (!__is_same(Tag, B16)) acc[it] = mfma16x16x32<B16>(th, lo, acc[it]);
      }
    }
    // in the layout of an accumulator: column lane & 15, tokens 4 (lane >> 4) ..
#pragma unroll
    for (int it = 0; it < 4; ++it) *((f32x4 *)(ws + (lay.u0 + ct * 4 + it) * 1024) + lane) = acc[it];
  }
}

// (reads that a barrier has waited for: the registers count as written here)
__device__ __forceinline__ void lds_landed(u32x4 &a) { asm volatile("" : "+v"(a)); }
__device__ __forceinline__ void lds_landed(u32x4 &a, u32x4 &b) { asm volatile("" : "+v"(a), "+v"(b)); }

// segments of `len` tokens: what they add to the state ahead of them [slot][heads][n * p], what becomes of that state: a product whose diagonal
// stays fp32 [slot][heads][n], the rest [slot][heads] (n x n as operands); the states that sequences of several segments come with [sequence][heads][n * p]; a sequence's slots
// start at cu_q / len + its number
struct Segments {
  float *added, *first, *diagonal;
  char *carry;
  int len;
};
enum { WHOLE, SEGMENTS, ADDED, CARRY };   // workgroups are sequences, or segments; ADDED, CARRY: only what a segment does to the state

// Workgroup = 4 waves x CW tiles of 16 columns of one head of one sequence; a wave keeps S of its columns in accumulators.  The
// accumulators are the next product's operands as they are: the rows of S are dealt so that tiles 2 s and 2 s + 1 together hold
// n = 32 s + 8 g .. + 7 in lane group g.  O is computed transposed (columns by tokens), so that a lane stores four columns of a token.
// Bound by the chain of a chunk and by the way of its 129 KB through the memory pipeline of a CU.  LDS holds one chunk, in groups in the order of their
// use: as soon as all waves have used a group, its part of the next chunk is asked for, so that transfers run all the time and none is waited for
// that was not asked for a chunk before (3 sequences of 4011 tokens and less, 8 heads of 128 x 128: 283 us with two phases, each fetched as a whole
// while the other was used, 247 with operands read as they were used -> 224).
// Few long sequences leave most CUs idle in it, and are cut into segments of whole chunks (pick_segment).  What a segment does to the state ahead
// of it is linear, S <- M S + C: a first launch walks the segments for C (from zeros, or what the sequence comes with) and M (from the identity, without
// values), with neither q nor B; the second starts a segment from the state that the C and M of those before it give, and is otherwise the walk.  Of the
// sequences above: 223 -> 54 + 63 us (11 chunks a segment; 5 - 8 times as many workgroups as sequences, heads and halves of them).
template <typename Tag, int NK, int CW, int MODE>
__device__ __forceinline__ void walk(const DeltaPrep &q, const Segments &sg, int wide, int at_head) {
  typedef typename elem<Tag>::T T;
  constexpr bool OUT = MODE == WHOLE || MODE == SEGMENTS, VALUES = MODE != CARRY;
  // fragments of W, Q and U0; steps of W and Q (U0 in the first) | B, decay | pairs of tiles of K
  constexpr int QF = OUT ? 8 * NK : 0, BF = OUT ? 16 : 0, F1 = 8 * NK + QF + (VALUES ? 16 * CW : 0), GROUPS = 2 * NK + 1;
  // transfers of a wave: for a group, for those behind it, for all
  constexpr int STEP = OUT ? 4 : 2, MIDDLE = OUT ? 5 : 1;
  constexpr auto own = [](int n) { return n < NK ? (n || !VALUES ? STEP : STEP + 4 * CW) : n == NK ? MIDDLE : 2; };
  constexpr auto behind = [](int n) { return n < NK ? STEP * (NK - 1 - n) + MIDDLE + 2 * NK : 2 * (GROUPS - 1 - n); };
  constexpr int ALL = own(0) + behind(0);
  const MvDeltaArgs &p = q.a;
  extern __shared__ __attribute__((aligned(16))) char smem[];   // [F1][1 KiB] | K | B | decay
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4;
  const int head = at_head / wide, tiles = MODE == CARRY ? 2 * NK : p.p / 16, tile0 = (at_head - head * wide) * 4 * CW;
  int seq = blockIdx.z, from = 0, q0 = 0, len = 0, all = 0;
  if constexpr (MODE == WHOLE) {
    q0 = p.cu_q[seq], all = len = p.cu_q[seq + 1] - q0;
  } else {
    seq = 0;
    for (int hi = p.n_seqs; hi - seq > 1;) {   // the sequence that the slot belongs to
      const int mid = (seq + hi) >> 1;
      if (p.cu_q[mid] / sg.len + mid <= (int)blockIdx.z) seq = mid;
      else hi = mid;
    }
    q0 = p.cu_q[seq], all = p.cu_q[seq + 1] - q0;
    from = ((int)blockIdx.z - q0 / sg.len - seq) * sg.len;
    len = min(sg.len, all - from);
    // (nobody asks for what the last one adds, nor for what becomes of the state ahead of the first)
    if (from < 0 || (!OUT && from + sg.len >= all) || (MODE == CARRY && from == 0)) return;
  }
  if (len <= 0) return;
  const int before = p.cu_k[seq + 1] - p.cu_k[seq] - all, slot = p.state_slots[seq];
  const bool keep = slot >= 0 && slot < p.slots;
  const int64_t size = (int64_t)p.heads * p.n * p.p;
  const Layout lay(NK, p.p);
  const int64_t stride = (int64_t)p.heads * lay.total * 1024;
  const char *ws = q.ws + ((int64_t)(q0 / L + seq + from / L) * p.heads + head) * lay.total * 1024 + lane * 16;
  q0 += from;

  int col[CW];
  bool live[CW];
#pragma unroll
  for (int w = 0; w < CW; ++w) {
    const int t = tile0 + wave * CW + w;
    live[w] = t < tiles, col[w] = min(t, tiles - 1) * 16 + r16;
  }
  auto state_row = [&](int i, int e) { return (i >> 1) * 32 + g * 8 + (i & 1) * 4 + e; };
  auto in_head = [&](int w, int i, int e) { return ((int64_t)head * p.n + state_row(i, e)) * p.p + col[w]; };
  auto state_at = [&](int half, int w, int i, int e) { return p.state + half * p.slots * size + (int64_t)(keep ? slot : 0) * size + in_head(w, i, e); };
  f32x4 st[CW][2 * NK];

  auto fetch = [&](const char *from, int frag, char *to) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(from + (int64_t)frag * 1024),
                                     (__attribute__((address_space(3))) void *)to, 16, 0, 0);
  };
  auto fetch_group = [&](auto G, int c) __attribute__((always_inline)) {
    constexpr int n = decltype(G)::value;
    const char *from = ws + c * stride;
    if constexpr (n < NK) {
#pragma unroll
      for (int i = 0; i < STEP; ++i) {   // (W's eight, then Q's)
        const int which = i * 4 + wave, f = (which >> 3) * 8 * NK + (((which >> 1) & 3) * NK + n) * 2 + (which & 1);
        fetch(from, f, smem + f * 1024);
      }
      if constexpr (n == 0 && VALUES) {
#pragma unroll
        for (int i = 0; i < 4 * CW; ++i) {
          const int f = i * 4 + wave;   // (column tile, token tile)
          fetch(from, lay.u0 + min(tile0 + (f >> 2), tiles - 1) * 4 + (f & 3), smem + (8 * NK + QF + f) * 1024);
        }
      }
    } else if constexpr (n == NK && !OUT) {
      fetch(from, lay.tail, smem + (F1 + 8 * NK) * 1024);   // (every wave: the same bytes)
    } else {
      constexpr int first = n == NK ? 8 * NK : (n - NK - 1) * 8, last = n == NK ? 8 * NK + 16 : first + 7;
#pragma unroll
      for (int i = 0; i < own(n); ++i) {
        const int f = min(first + i * 4 + wave, last);
        fetch(from, lay.k + f, smem + (F1 + f) * 1024);
      }
    }
  };
  const uint32_t base = lds_address(smem) + lane * 16;   // (fragments)
  const uint32_t aw = base, aq = base + 8 * NK * 1024, au = base + (8 * NK + QF + wave * CW * 4) * 1024;
  const uint32_t ak = base + F1 * 1024, ab = ak + 8 * NK * 1024, at = lds_address(smem) + (F1 + 8 * NK + BF) * 1024 + g * 32;
  const int chunks = (len + L - 1) / L;
  const bool quads = !(((uintptr_t)p.out & 7) | (p.out_stride & 3));   // (rows of the output may stand anywhere)
  if constexpr (MODE != SEGMENTS) static_for<GROUPS>([&](auto G) { fetch_group(G, 0); });

  // ---- the state ahead
  const int64_t first_at = (int64_t)seq * size;
#pragma unroll
  for (int w = 0; w < CW; ++w)
#pragma unroll
    for (int i = 0; i < 2 * NK; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = 0.f;
        if constexpr (MODE == CARRY) {
          v = state_row(i, e) == col[w] ? 1.f : 0.f;
        } else if (from == 0 && keep && before > 0) {
          // (the pool's state of a cut sequence is read by the first launch alone: the second may write it)
          v = MODE == SEGMENTS && all > len ? sg.first[first_at + in_head(w, i, e)] : *state_at(before & 1, w, i, e);
        }
        if (MODE == ADDED && from == 0 && before > 0 && live[w]) sg.first[first_at + in_head(w, i, e)] = v;
        st[w][i][e] = v;
      }
  if constexpr (MODE == SEGMENTS) {
    // .. of a later segment: that at the end of the first, and from segment to segment one product, whose left operand lands in LDS while
    // the one before is multiplied (where LDS holds two: up to 128 channels).  Read by each wave as it was used, a segment took 4.5 us.
    // Within a segment the state crosses chunks in fp32 (S *= decay), and so that no more is lost from segment to segment, M's diagonal stays in fp32 and
    // the product of the rests is not left out: the kept states are as far from 64 bits as those of whole sequences (0.999 of it over 60 shapes, lengths
    // and decays; with all of M in two bf16 numbers and three products up to 1.10, where nothing decays).  That costs 1.5 of 248 us.
    constexpr int CF = 4 * NK * NK, BUFFERS = 2 * CF <= F1 + 8 * NK + BF + 1 ? 2 : 1;   // fragments
    const int ahead = from / sg.len, first = (int)blockIdx.z - ahead;
    auto fetch_carry = [&](int j) __attribute__((always_inline)) {
      const char *of = sg.carry + ((int64_t)(first + j) * p.heads + head) * (CF * 1024) + lane * 16;
#pragma unroll
      for (int i = 0; i < NK * NK; ++i) fetch(of, i * 4 + wave, smem + ((j % BUFFERS) * CF + i * 4 + wave) * 1024);
    };
    f32x4 next[CW][2 * NK], diagonal[2 * NK];
    auto load_added = [&](int j) __attribute__((always_inline)) {
#pragma unroll
      for (int w = 0; w < CW; ++w)
#pragma unroll
        for (int i = 0; i < 2 * NK; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) next[w][i][e] = sg.added[(first + j) * size + in_head(w, i, e)];
#pragma unroll
      for (int i = 0; i < 2 * NK; ++i)
        if (j > 0) diagonal[i] = *(const f32x4 *)(sg.diagonal + ((int64_t)(first + j) * p.heads + head) * p.n + state_row(i, 0));
    };
    if (ahead > 0) {
      if (ahead > 1) fetch_carry(1);
      load_added(0);
#pragma unroll
      for (int w = 0; w < CW; ++w)
#pragma unroll
        for (int i = 0; i < 2 * NK; ++i) st[w][i] = next[w][i];
      if (ahead > 1) load_added(1);
      for (int j = 1; j < ahead; ++j) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
        u32x4 sh[CW][NK], sl[CW][NK], f[2][NK][2];
#pragma unroll
        for (int w = 0; w < CW; ++w) {
#pragma unroll
          for (int s = 0; s < NK; ++s) split44(st[w][2 * s], st[w][2 * s + 1], sh[w][s], sl[w][s]);
#pragma unroll
          for (int i = 0; i < 2 * NK; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) st[w][i][e] = fmaf(diagonal[i][e], st[w][i][e], next[w][i][e]);
        }
        if (j + 1 < ahead) {
          if constexpr (BUFFERS == 2) fetch_carry(j + 1);
          load_added(j + 1);
        }
        const uint32_t left = base + (j % BUFFERS) * CF * 1024;
        auto read_tile = [&](auto I) __attribute__((always_inline)) {
          constexpr int i = decltype(I)::value;
          static_for<2 * NK>([&](auto M) {
            constexpr int m = decltype(M)::value;
            lds_read128<m * 1024>(f[i & 1][m >> 1][m & 1], left + i * NK * 2048);
          });
        };
        read_tile(std::integral_constant<int, 0>{});
        static_for<2 * NK>([&](auto I) {
          constexpr int i = decltype(I)::value;
          static_for<NK>([&](auto S) { lds_wait<0>(f[i & 1][decltype(S)::value][0], f[i & 1][decltype(S)::value][1]); });
          if constexpr (i + 1 < 2 * NK) read_tile(std::integral_constant<int, i + 1>{});
          f32x4 half[CW];   // (two sums: a product waits for the one before it)
#pragma unroll
          for (int w = 0; w < CW; ++w) half[w] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int part = 0; part < 4; ++part)
#pragma unroll
            for (int s = 0; s < NK; ++s)
#pragma unroll
              for (int w = 0; w < CW; ++w) {
                f32x4 &to = (part * NK + s) & 1 ? half[w] : st[w][i];
                to = mfma16x16x32<B16>(f[i & 1][s][part >= 2], part & 1 ? sl[w][s] : sh[w][s], to);
              }
#pragma unroll
          for (int w = 0; w < CW; ++w) st[w][i] += half[w];
        });
        if (BUFFERS == 1 && j + 1 < ahead) {
          lds_barrier();
          fetch_carry(j + 1);
        }
      }
      lds_barrier();
    }
    static_for<GROUPS>([&](auto G) { fetch_group(G, 0); });
  }

  for (int c = 0; c < chunks; ++c) {
    const bool more = c + 1 < chunks;
    // Before a group is used: it has landed (the transfers of the others may be under way; stores only make the wait longer), and every wave is done
    // with the group before, whose place the next chunk's takes.
    auto begin = [&](auto G) __attribute__((always_inline)) {
      constexpr int n = decltype(G)::value;
      if (n == 0 || more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(ALL - own(n) - own((n + GROUPS - 1) % GROUPS)) : "memory");
      else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(behind(n)) : "memory");
      lds_barrier();
      if constexpr (n == 0) {
        if (c > 0) fetch_group(std::integral_constant<int, GROUPS - 1>{}, c);
      } else {
        if (more) fetch_group(std::integral_constant<int, n - 1>{}, c + 1);
      }
    };
    // The operands of a group are read while the products of the one before run.
    u32x4 fw[2][4][2], fo[2][4][2], u0[CW][4], fb[kTriangle][2], tail[2 * NK], fk[2][2][2][2];
    auto read_step = [&](auto S) __attribute__((always_inline)) {
      constexpr int s = decltype(S)::value;
      static_for<4>([&](auto I) {
        constexpr int it = decltype(I)::value;
        static_for<2>([&](auto P) {
          constexpr int h = decltype(P)::value;
          lds_read128<((it * NK + s) * 2 + h) * 1024>(fw[s & 1][it][h], aw);
          if constexpr (OUT) lds_read128<((it * NK + s) * 2 + h) * 1024>(fo[s & 1][it][h], aq);
        });
      });
    };
    auto read_pair = [&](auto P) __attribute__((always_inline)) {
      constexpr int pair = decltype(P)::value;
      static_for<8>([&](auto I) {
        constexpr int i = decltype(I)::value;
        lds_read128<(pair * 8 + i) * 1024>(fk[pair & 1][i >> 2][(i >> 1) & 1][i & 1], ak);
      });
    };
    auto begin_step = [&](auto N) __attribute__((always_inline)) {   // the group behind the one that is about to be multiplied
      constexpr int n = decltype(N)::value;
      begin(N);
      if constexpr (n < NK) {
        read_step(N);
      } else if constexpr (n == NK) {
        static_for<(OUT ? kTriangle : 0)>([&](auto M) {
          constexpr int m = decltype(M)::value, it = m < 2 ? m : m / 2 + 1, s = m < 2 ? 0 : m % 2;
          lds_read128<((it * 2 + s) * 2) * 1024>(fb[m][0], ab);
          lds_read128<((it * 2 + s) * 2 + 1) * 1024>(fb[m][1], ab);
        });
        static_for<2 * NK>([&](auto I) { lds_read128<(decltype(I)::value >> 1) * 128 + (decltype(I)::value & 1) * 16>(tail[decltype(I)::value], at); });
      } else {
        read_pair(std::integral_constant<int, n - NK - 1>{});
      }
    };
    begin(std::integral_constant<int, 0>{});
    static_for<(VALUES ? 4 * CW : 0)>([&](auto I) { lds_read128<decltype(I)::value * 1024>(u0[decltype(I)::value / 4][decltype(I)::value % 4], au); });
    read_step(std::integral_constant<int, 0>{});
    // ---- U = U0 - W S, O = Q S
    f32x4 u[CW][4], o[CW][4];
    static_for<NK>([&](auto S) {
      constexpr int s = decltype(S)::value;
      u32x4 sh[CW], sl[CW];
#pragma unroll
      for (int w = 0; w < CW; ++w) split44(st[w][2 * s], st[w][2 * s + 1], sh[w], sl[w]);
      begin_step(std::integral_constant<int, s + 1>{});   // (its barrier comes behind all reads of this group)
      static_for<4>([&](auto I) {
        constexpr int it = decltype(I)::value;
        lds_landed(fw[s & 1][it][0], fw[s & 1][it][1]);
        if constexpr (OUT) lds_landed(fo[s & 1][it][0], fo[s & 1][it][1]);
      });
      if constexpr (s == 0)
        static_for<4 * CW>([&](auto I) {
          constexpr int w = decltype(I)::value / 4, it = decltype(I)::value % 4;
          o[w][it] = u[w][it] = f32x4{0.f, 0.f, 0.f, 0.f};
          if constexpr (VALUES) {
            lds_landed(u0[w][it]);
            u[w][it] = __builtin_bit_cast(f32x4, u0[w][it]);
          }
        });
#pragma unroll
      for (int part = 0; part < 3; ++part)
#pragma unroll
        for (int it = 0; it < 4; ++it)
#pragma unroll
          for (int w = 0; w < CW; ++w) {
            u[w][it] = mfma16x16x32<B16>(fw[s & 1][it][part == 2], part == 1 ? sl[w] : sh[w], u[w][it]);
            if constexpr (OUT) o[w][it] = mfma16x16x32<B16>(part == 1 ? sl[w] : sh[w], fo[s & 1][it][part == 2], o[w][it]);
          }
    });
    // ---- O += B U, S = decay S + K U
    u32x4 uh[CW][2], ul[CW][2];
#pragma unroll
    for (int w = 0; w < CW; ++w)
#pragma unroll
      for (int s = 0; s < 2; ++s) split44(u[w][2 * s], u[w][2 * s + 1], uh[w][s], ul[w][s]);
    begin_step(std::integral_constant<int, NK + 1>{});
    static_for<(OUT ? kTriangle : 0)>([&](auto M) { lds_landed(fb[decltype(M)::value][0], fb[decltype(M)::value][1]); });
    static_for<2 * NK>([&](auto I) {
      constexpr int i = decltype(I)::value;
      lds_landed(tail[i]);
#pragma unroll
      for (int w = 0; w < CW; ++w) st[w][i] *= __builtin_bit_cast(f32x4, tail[i]);
    });
    if constexpr (OUT) {
      static_for<4>([&](auto I) {
        constexpr int it = decltype(I)::value;
#pragma unroll
        for (int part = 0; part < 3; ++part)
          static_for<it / 2 + 1>([&](auto S) {
            constexpr int s = decltype(S)::value;
#pragma unroll
            for (int w = 0; w < CW; ++w)
              o[w][it] = mfma16x16x32<B16>(part == 1 ? ul[w][s] : uh[w][s], fb[triangle(it, s)][part == 2], o[w][it]);
          });
      });
#pragma unroll
      for (int w = 0; w < CW; ++w)
#pragma unroll
        for (int it = 0; it < 4; ++it) {
          const int t = c * L + 16 * it + r16;
          T *to = (T *)p.out + (int64_t)(q0 + t) * p.out_stride + head * p.p + col[w] - r16 + 4 * g;
          if (!live[w] || t >= len) continue;
          if (quads) {
            *(u32x2 *)to = pack_quad<Tag>(o[w][it]);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) to[e] = elem<Tag>::st(o[w][it][e]);
          }
        }
    }
    static_for<NK>([&](auto P) {   // two state tiles at a time
      constexpr int pair = decltype(P)::value, i0 = 2 * pair;
      if constexpr (pair + 1 < NK) begin_step(std::integral_constant<int, NK + 2 + pair>{});
      else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      static_for<2>([&](auto D) {
        constexpr int d = decltype(D)::value;
        lds_landed(fk[pair & 1][d][0][0], fk[pair & 1][d][0][1]);
        lds_landed(fk[pair & 1][d][1][0], fk[pair & 1][d][1][1]);
      });
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int part = 0; part < 3; ++part)
#pragma unroll
          for (int d = 0; d < 2; ++d)
#pragma unroll
            for (int w = 0; w < CW; ++w)
              st[w][i0 + d] = mfma16x16x32<B16>(fk[pair & 1][d][s][part == 2], part == 1 ? ul[w][s] : uh[w][s], st[w][i0 + d]);
    });
  }
  if constexpr (MODE == ADDED) {
#pragma unroll
    for (int w = 0; w < CW; ++w)
      if (live[w]) {
#pragma unroll
        for (int i = 0; i < 2 * NK; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) sg.added[(int64_t)blockIdx.z * size + in_head(w, i, e)] = st[w][i][e];
      }
  } else if constexpr (MODE == CARRY) {
    // by rows through LDS: the left operand of the product with the state ahead, in the order of its accumulators
    constexpr int CS = 64 * CW + 4;   // row stride
    float *cs = (float *)smem;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < CW; ++w)
#pragma unroll
      for (int i = 0; i < 2 * NK; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool diagonal = live[w] && state_row(i, e) == col[w];
          if (diagonal) sg.diagonal[((int64_t)blockIdx.z * p.heads + head) * p.n + col[w]] = st[w][i][e];
          cs[state_row(i, e) * CS + (wave * CW + w) * 16 + r16] = diagonal ? 0.f : st[w][i][e];
        }
    __syncthreads();
    char *carry = sg.carry + ((int64_t)blockIdx.z * p.heads + head) * (4 * NK * NK * 1024) + lane * 16;
    for (int f = wave; f < 2 * NK * 2 * CW; f += 4) {
      const int i = f / (2 * CW), s = f - i * (2 * CW), to = tile0 / 2 + s;
      if (to >= NK) continue;
      const float *row = cs + ((i >> 1) * 32 + (r16 >> 2) * 8 + (i & 1) * 4 + (r16 & 3)) * CS + 32 * s + 8 * g;
      u32x4 hi, lo;
      split44(*(const f32x4 *)row, *(const f32x4 *)(row + 4), hi, lo);
      *(u32x4 *)(carry + ((i * NK + to) * 2) * 1024) = hi;
      *(u32x4 *)(carry + ((i * NK + to) * 2 + 1) * 1024) = lo;
    }
  } else if (keep && from + len >= all) {
#pragma unroll
    for (int w = 0; w < CW; ++w)
      if (live[w]) {
#pragma unroll
        for (int i = 0; i < 2 * NK; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) *state_at((before + all) & 1, w, i, e) = st[w][i][e];
      }
  }
}

// (workgroups are dealt to the 8 XCDs in turn: each gets a run of columns and heads, which share all but their part of U0)
__device__ __forceinline__ int by_xcd(int wide, int heads) {
  const int all = wide * heads, at = blockIdx.y * wide + blockIdx.x;
  return all & 7 ? at : (at & 7) * (all >> 3) + (at >> 3);
}
template <typename Tag, int NK, int CW, int MODE>
__global__ void __launch_bounds__(256, 1) delta_walk_kernel(DeltaPrep q, Segments sg) {
  walk<Tag, NK, CW, MODE>(q, sg, gridDim.x, by_xcd(gridDim.x, q.a.heads));
}
// what the segments add, and what becomes of the state ahead of them: workgroups of either beside each other
template <typename Tag, int NK, int CW>
__global__ void __launch_bounds__(256, 1) delta_segments_kernel(DeltaPrep q, Segments sg, int added) {
  const int wide = gridDim.x, at = by_xcd(wide, q.a.heads), head = at / wide, x = at - head * wide;
  if (x < added) walk<Tag, NK, CW, ADDED>(q, sg, added, head * added + x);
  else walk<Tag, NK, CW, CARRY>(q, sg, wide - added, head * (wide - added) + x - added);
}

inline int64_t segment_slots(int n_seqs, int total_q, int seg) { return (int64_t)total_q / (seg * L) + n_seqs; }
// Chunks of a segment; 0: whole sequences.  A chunk of a whole sequence being 1, one of both launches is 2.1 (3 of 32 key channels), a product with the state ahead 0.6 and
// the second launch 2.5; a segment of the square root of a third of the longest is the shortest way through both, and there are to be no more
// workgroups than CUs (each holds one: rounds behind the first cost what they save).  us of the whole call, whole and cut; n x p, heads x sequences:
//   128 x 128: 4 x 1, 8 chunks 54 and 53, 12: 68 and 58, 24: 115 and 76, 63: 249 and 97; 8 x 3 (the later ones shorter), 24: 122 and 90, 63: 317 and 199;
//   16 x 3, 12: 82 and 85, 24: 155 and 153, 63: 411 and 382.    64 x 64: 16 x 1, 12: 50 and 42, 63: 177 and 84; 16 x 3, 24: 95 and 77.
//   32 x 128: 4 x 10 of 2148 tokens at most 106 and 112.   160 x 128: 8 x 1, 24: 136 and 93; 16 x 3, 24: 219 and 219.   128 x 256: 16 x 1, 24: 123 and 103; 16 x 3, 63: 433 and 524.
// A sequence's segments, and so the last bits of its results, depend on the call's other sequences; a whole sequence has the same bits in any call.
inline int pick_segment(int n_seqs, int total_q, int max_q, int heads, int p, int n) {
  const int tiles = p / 16, workgroups = std::max((tiles + 3) / 4, (tiles + 7) / 8 + (n / 16 + 7) / 8) * heads;   // (of either launch)
  const int64_t longest = ((int64_t)max_q + L - 1) / L, chunks = ((int64_t)total_q + L - 1) / L;
  const int64_t room = 256 - (int64_t)n_seqs * workgroups / 2;   // (a sequence's last segment is half a segment)
  if (room <= 0) return 0;
  const int64_t seg = std::max<int64_t>({2, (int64_t)std::ceil(std::sqrt(longest / 3.0)), (chunks * workgroups + room - 1) / room});
  return (n > 32 ? 2.1 : 3.0) * seg + 0.6 * longest / seg + 2.5 < longest ? (int)seg : 0;
}

template <typename Tag, int NK>
int launch(const DeltaPrep &q, int seg, hipStream_t stream) {
  const MvDeltaArgs &a = q.a;
  constexpr int RS = NK * 32 + 4, KS = NK * 32 + 8;
  constexpr int QB = L * KS * 2 > L * (L + 4) * 4 ? L * KS * 2 : L * (L + 4) * 4;
  const dim3 grid((unsigned)chunk_slots(a.n_seqs, a.total_q), a.heads), block(kPrepareWaves * 64);
  constexpr int need = L * RS * 4 + L * KS * 2 + QB + (3 + kPrepareWaves) * L * 4;
  if (q.raw) {
    if (int rc = mv_allow_lds<delta_prepare_kernel<Tag, NK, true>>()) return rc;
    hipLaunchKernelGGL((delta_prepare_kernel<Tag, NK, true>), grid, block, need, stream, q);
  } else {
    if (int rc = mv_allow_lds<delta_prepare_kernel<Tag, NK, false>>()) return rc;
    hipLaunchKernelGGL((delta_prepare_kernel<Tag, NK, false>), grid, block, need, stream, q);
  }
  MV_LAUNCH_CHECK();
  const int tiles = a.p / 16, wide = (tiles + 7) / 8, narrow = (tiles + 3) / 4;
  constexpr auto lds = [](int columns) { return (24 * NK + 16 * columns + 17) * 1024; };
  if (seg) {
    Segments sg;
    sg.len = seg * L;
    const int64_t slots = segment_slots(a.n_seqs, a.total_q, seg), state = (int64_t)a.heads * a.n * a.p;
    sg.added = (float *)(q.ws + mv_delta_chunk_workspace(a.n_seqs, a.total_q, a.heads, a.p, a.n));
    sg.first = sg.added + slots * state, sg.diagonal = sg.first + a.n_seqs * state, sg.carry = (char *)(sg.diagonal + slots * a.heads * a.n);
    const int carried = (2 * NK + 7) / 8, by_rows = 32 * NK * (64 * 2 + 4) * 4;
    const int need = std::max((16 * NK + 32 + 1) * 1024, by_rows);
    if (int rc = mv_allow_lds<delta_segments_kernel<Tag, NK, 2>>()) return rc;
    hipLaunchKernelGGL((delta_segments_kernel<Tag, NK, 2>), dim3(wide + carried, a.heads, (unsigned)slots), dim3(256), need, stream, q, sg, wide);
    MV_LAUNCH_CHECK();
    if (int rc = mv_allow_lds<delta_walk_kernel<Tag, NK, 1, SEGMENTS>>()) return rc;
    hipLaunchKernelGGL((delta_walk_kernel<Tag, NK, 1, SEGMENTS>), dim3(narrow, a.heads, (unsigned)slots), dim3(256), lds(1), stream, q, sg);
    MV_LAUNCH_CHECK();
    return MV_OK;
  }
  // two column tiles a wave share every operand read, where that still leaves a workgroup per CU and LDS holds their chunk (up to 128 channels)
  if constexpr (lds(2) <= 160 * 1024) {
    if (tiles > 4 && (int64_t)wide * a.heads * a.n_seqs >= 256) {
      if (int rc = mv_allow_lds<delta_walk_kernel<Tag, NK, 2, WHOLE>>()) return rc;
      hipLaunchKernelGGL((delta_walk_kernel<Tag, NK, 2, WHOLE>), dim3(wide, a.heads, a.n_seqs), dim3(256), lds(2), stream, q, Segments{});
      MV_LAUNCH_CHECK();
      return MV_OK;
    }
  }
  if (int rc = mv_allow_lds<delta_walk_kernel<Tag, NK, 1, WHOLE>>()) return rc;
  hipLaunchKernelGGL((delta_walk_kernel<Tag, NK, 1, WHOLE>), dim3(narrow, a.heads, a.n_seqs), dim3(256), lds(1), stream, q, Segments{});
  MV_LAUNCH_CHECK();
  return MV_OK;
}

// bf16, one decay per head: whether the convolution along with the preparation is the shorter way.  Its pieces (four channels, eight tokens) are one turn of a workgroup's
// threads or several, each a trip to memory of its own, where the convolution's own launch has a piece to a thread; chunks beside each other on a CU cover that, and
// short prompts of up to two turns are the host's, for whom it is a launch less (beyond, the GPU loses more than the host gains).  us along / apart by workgroups:
//   two heads of 64 x 64 (one turn): 6 22.0 / 22.9, 496 37.0 / 39.0; of 64 x 32 (one turn; why is not known): 1656 174 / 176, 2512 137 / 134, 5024 265 / 254
//   two heads of 128 x 128 (two turns), in a graph: 8 22.9 / 21.4, 68 32.6 / 31.1, 84 56.4 / 55.3, 136 39.2 / 39.7, 736 72.5 / 73.5; the layer around them: 1 x 64 tokens
//   34.1 / 36.2, 2 x 239 34.4 / 36.9, 1 x 281 36.2 and 37.5 / 37.0 and 36.5, 2 x 400 43.1 / 41.6
//   two heads of 256 x 128 (three): 40 54.5 / 50.1, 1096 193.8 / 190.6
//   one head of 128 x 32 (1.5): 28 26.6 / 25.3; of 64 x 64 (1.5): 198 73.1 / 75.1, 2512 113.5 / 121.6; of 128 x 128 (three): 48 24.3 / 21.5, 200 30.9 / 29.1,
//   404 54.4 / 56.2, 992 73.1 / 79.2; four turns: 296 80.6 / 78.5
bool conv_along(const MvDeltaArgs &a) {
  const int of_group = a.heads / a.groups;
  const int64_t threads = 256 * of_group, pieces = (2 * a.n + of_group * a.p) / 4 * (L / 8), groups = chunk_slots(a.n_seqs, a.total_q) * a.groups;
  if (pieces <= threads) return of_group == 1 || a.n > 32 || groups <= 2000;
  if (pieces <= 2 * threads && a.max_q * pieces <= 512 * threads) return true;
  return 2 * pieces <= (of_group == 1 ? 7 : 4) * threads && groups * threads >= 120 * (pieces - threads);
}

}  // namespace

// The convolution goes along where every channel is one workgroup's (which reads and writes what is kept of it), a thread's window is the taps (in one of more, an
// infinite input times a weight that is not there would reach tokens that it does not belong to) and, with a head's values prepared (not bf16 with one decay
// per head), a wave has one tile of them and LDS holds them in the decays' place
bool mv_delta_chunk_takes_conv(const MvDeltaArgs &a, int dtype) {
  const bool scalar = dtype == MV_BF16 && !a.channel_decay;
  const int of_group = a.heads / a.groups;
  return (scalar ? of_group <= 2 && conv_along(a) : of_group == 1 && a.p <= 16 * kPrepareWaves && a.p <= 2 * a.n) && a.taps == kChunkTaps &&
         a.k_off == a.heads * a.p && a.q_off == a.k_off + a.groups * a.n && a.channels == a.q_off + a.groups * a.n;
}

size_t mv_delta_chunk_workspace(int n_seqs, int total_q, int heads, int p, int n) {
  if (n_seqs <= 0 || total_q <= 0 || heads <= 0 || p <= 0 || n <= 0 || n > 160 || (n & 31)) return 0;
  return (size_t)chunk_slots(n_seqs, total_q) * heads * Layout(n / 32, p).total * 1024;
}

// (behind the above)
size_t mv_delta_segments_workspace(int n_seqs, int total_q, int max_q, int heads, int p, int n) {
  if (max_q <= MV_DELTA_WHOLE || !mv_delta_chunk_workspace(n_seqs, total_q, heads, p, n)) return 0;
  const int seg = pick_segment(n_seqs, total_q, max_q, heads, p, n);
  if (!seg) return 0;
  const int64_t slots = segment_slots(n_seqs, total_q, seg);
  if (slots > 65535) return 0;
  return ((slots + n_seqs) * p + slots + slots * n) * (size_t)heads * n * 4;
}

int mv_delta_chunk_launch(const MvDeltaArgs &a, const void *raw, int64_t raw_stride, int dtype, bool *normed, hipStream_t stream) {
  const size_t need = mv_delta_chunk_workspace(a.n_seqs, a.total_q, a.heads, a.p, a.n);
  if (!need || !a.workspace) return MV_E_SHAPE;   // larger states: token by token
  if ((size_t)a.ws_bytes < need || !mv_aligned16(a.workspace)) return MV_E_WORKSPACE;
  if (!mv_aligned16(a.x) || (a.x_stride & 7) || (a.k_off & 7) || (a.q_off & 7) || a.total_q > 64 * 1000000) return MV_E_ALIGN;
  if (a.channel_decay && (!mv_aligned16(a.a) || (a.a_stride & 7) || !mv_aligned16(a.dt_bias))) return MV_E_ALIGN;
  const DeltaPrep q{a, (char *)a.workspace, raw, raw_stride};
  if (!a.channel_decay && dtype == MV_BF16) return mv_delta_scalar_launch(a, raw, raw_stride, normed, stream);
  if (normed) *normed = false;
  const size_t more = mv_delta_segments_workspace(a.n_seqs, a.total_q, a.max_q, a.heads, a.p, a.n);
  const int seg = more && (size_t)a.ws_bytes >= need + more ? pick_segment(a.n_seqs, a.total_q, a.max_q, a.heads, a.p, a.n) : 0;
#define MV_DN(NK_) \
  if (a.n == 32 * NK_) return dtype == MV_BF16 ? launch<bf16_tag, NK_>(q, seg, stream) : launch<f16_tag, NK_>(q, seg, stream)
  MV_DN(1);
  MV_DN(2);
  MV_DN(3);
  MV_DN(4);
  MV_DN(5);
#undef MV_DN
  return MV_E_SHAPE;
}
