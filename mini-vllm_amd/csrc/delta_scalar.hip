// K16 — gated delta rule of prompts in chunks where a head has one decay (bf16 operands, fp32 state).
//
// With r_i the running sum of the log decays in a chunk, the decays leave the products over channels: with the factors f_i, g_i that scale k
// and q to their lengths, S the state ahead of the chunk and T as in delta_chunk.hip,
//     A_ij = beta_i f_i f_j e^{r_i - r_j} (k_i k_j)      U = T R,  R_i = v_i - e^{r_i} f_i (k_i S)
//     B_ij = g_i f_j e^{r_i - r_j} (q_i k_j)             o_i = e^{r_i} g_i (q_i S) + sum_{j <= i} B_ij u_j
//     S <- e^{r_last} S + sum_j k_j (e^{r_last - r_j} f_j u_j)^T
// so k and q enter every product as they are in memory (exact in bf16) and only T, B, S and U are sums of two bf16 numbers.  Two launches:
//   prepare: T, B and three factors per token, one workgroup per (chunk, pair of heads with the same k and q), 25 KiB of workspace a head;
//   walk:    chunks one behind the other, one workgroup per (sequence, head, columns); rows of k, q and v come from the inputs, transposed out of
//            LDS where the state takes them in; the next chunk lands while this one is multiplied.
#include "delta_chunk.h"

namespace {

// workspace of a (chunk, head) in fragments of 1 KiB: T [kTriangle][high, rest] | B [kTriangle][high, rest] | factors
constexpr int kB = 2 * kTriangle, kFactors = 4 * kTriangle, kScalarTotal = kFactors + 1;

// where 8 channels of a row lie in a fragment of 16 rows x 32 channels: four adjacent lanes of the transfer hold one row's 64 bytes, in an
// order that spreads the rows over the banks
__device__ __forceinline__ int row_chunk(int lane) { return (lane & 3) ^ ((lane >> 4) & 3); }
__device__ __forceinline__ int row_place(int row, int chunk) { return row * 4 + (chunk ^ ((row >> 2) & 3)); }

// Workgroup = HEADS heads of four waves each that share k and q of a chunk: the products k k^T and q k^T are theirs in common, decays, solution and results
// their own.  Bound by the latency of its phases, which 16 to 20 waves a CU cover in part: everything is asked for from memory at the start.
// CONV (q.raw: projected channels; a group's heads are this workgroup's): the causal convolution and silu of causal_conv_kernel (the same sums) ahead of it, four
// channels and eight tokens a thread and turn, into a.x, where the walk reads it, and k and q into LDS at once: a launch and a way of k and q through memory less.  Four
// channels, not eight: 80 registers leave three workgroups a CU, whose convolutions run beside the others' chains.  16 heads over 8 of 128 x 128, 16 sequences of up
// to 1490 tokens: 64 + 55 us as two launches, 120 with eight channels, 111 now (416 MB, 3.7 TB/s; a copy 4.7); the layer 248 -> 242.  Few tokens are the host's and a
// launch's: 70 tokens of one sequence 57 -> 33.
template <int NK, int HEADS, bool CONV>
__global__ void __launch_bounds__(256 * HEADS, CONV ? 6 : 4) delta_scalar_prepare_kernel(DeltaPrep q) {
  typedef uint16_t T;
  typedef elem<B16>::T E;
  constexpr int N = NK * 32, KS = N + 8, W = 4 * HEADS;   // LDS row stride
  const MvDeltaArgs &p = q.a;
  constexpr int QB = L * KS * 2 > L * TS * 4 ? L * KS * 2 : L * TS * 4, KB = HEADS > 1 ? QB : L * KS * 2;
  __shared__ __attribute__((aligned(16))) char smem[KB + QB + (2 + 2 * HEADS) * L * 4];
  T *ks = (T *)smem, *qs = (T *)(smem + KB);   // [L][KS]; later -A, then T, of the first head from qs on, of the second from ks on
  float *fk = (float *)(smem + KB + QB), *fq = fk + L, *bts = fq + L, *rss = bts + HEADS * L;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
  const int of = HEADS > 1 ? wave >> 2 : 0, head = blockIdx.y * HEADS + of;   // (of this wave)
  const int seq = chunk_sequence(p, blockIdx.x);
  const int q0 = p.cu_q[seq], len = p.cu_q[seq + 1] - q0, t0 = ((int)blockIdx.x - q0 / L - seq) * L;
  if (t0 >= len) return;
  const int nt = min(L, len - t0), grp = head / (p.heads / p.groups);
  char *ws = q.ws + ((int64_t)blockIdx.x * p.heads + head) * kScalarTotal * 1024;
  const T *x = (const T *)p.x + (int64_t)(q0 + t0) * p.x_stride;
  float *ts = (float *)(of ? (char *)ks : (char *)qs), *bt = bts + of * L, *rs = rss + of * L;

  // ---- k, q (tokens behind the end: zeros) and their lengths, four threads a token: both, or with two heads k by one half, q by the other (a length is
  // the same sum in either form); a head's first wave its betas and log2 decays, a lane a token
  {
    const int t = (tid & 255) >> 2, part = tid & 3;
    u32x4 a[NK], b[HEADS > 1 ? 1 : NK];
    if constexpr (!CONV) {
      const T *row = x + (int64_t)min(t, nt - 1) * p.x_stride + grp * N + part * 8;
#pragma unroll
      for (int i = 0; i < NK; ++i) {
        a[i] = *(const u32x4 *)(row + (of ? p.q_off : p.k_off) + 32 * i);
        if constexpr (HEADS == 1) b[i] = *(const u32x4 *)(row + p.q_off + 32 * i);
      }
    }
    const bool leads = (wave & 3) == 0;
    float beta = 0.f, decay = 0.f, bias = 0.f, rate = 0.f;
    if (leads) {
      const int64_t at = q0 + t0 + min(lane, nt - 1);
      beta = elem<B16>::ld(((const E *)p.beta)[at * p.beta_stride + head]), decay = elem<B16>::ld(((const E *)p.a)[at * p.a_stride + head]);
      rate = elem<B16>::ld(((const E *)p.a_log)[head]), bias = elem<B16>::ld(((const E *)p.dt_bias)[head]);
    }
    if constexpr (CONV) {
      T *xc = (T *)p.x + (int64_t)(q0 + t0) * p.x_stride;
      conv_chunk<B16, N, 256 * HEADS, false>(q, seq, q0, len, t0, nt, grp, blockIdx.y * HEADS * p.p, HEADS * p.p, tid, [&](int which, int row, int at, int c, u32x2 done) {
        if (row < nt) *(u32x2 *)(xc + (int64_t)row * p.x_stride + c) = done;
        if (which < 2) *(u32x2 *)((which ? qs : ks) + row * KS + at) = done;
      });
      __syncthreads();
#pragma unroll
      for (int i = 0; i < NK; ++i) {
        a[i] = *(const u32x4 *)((of ? qs : ks) + t * KS + part * 8 + 32 * i);
        if constexpr (HEADS == 1) b[i] = *(const u32x4 *)(qs + t * KS + part * 8 + 32 * i);
      }
    }
    auto length = [&](u32x4 *raw, T *to, float scale) {
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < NK; ++i) {
        if (t >= nt) raw[i] = u32x4{0u, 0u, 0u, 0u};
        float f[8];
        unpack8<B16>(raw[i], f);
#pragma unroll
        for (int j = 0; j < 8; ++j) sum = fmaf(f[j], f[j], sum);
        if constexpr (!CONV) *(u32x4 *)(to + t * KS + part * 8 + 32 * i) = raw[i];
      }
      return scale / sqrtf(lanes_sum<4>(sum) + p.unit_eps);
    };
    const float first = length(a, of ? qs : ks, of ? p.q_scale : 1.f);
    if (part == 0) (of ? fq : fk)[t] = first;
    if constexpr (HEADS == 1) {
      const float second = length(b, qs, p.q_scale);
      if (part == 0) fq[t] = second;
    }
    if (leads) {
      rate = -expf(rate) * 1.4426950408889634f;
      float sum = lane < nt ? rate * softplus_fast(decay + bias) : 0.f;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const float left = __shfl_up(sum, o, 64);
        if (lane >= o) sum += left;
      }
      rs[lane] = sum, bt[lane] = lane < nt ? sigmoid_f32(beta) : 0.f;
    }
  }
  __syncthreads();
  if ((wave & 3) == 0) {
    float *f = (float *)(ws + kFactors * 1024);
    const float last = rs[L - 1];
    const bool is = lane < nt;
    f[lane] = is ? fk[lane] * __builtin_amdgcn_exp2f(rs[lane]) : 0.f;
    f[L + lane] = is ? fq[lane] * __builtin_amdgcn_exp2f(rs[lane]) : 0.f;
    f[2 * L + lane] = is ? fk[lane] * __builtin_amdgcn_exp2f(last - rs[lane]) : 0.f;
    f[3 * L + lane] = __builtin_amdgcn_exp2f(last);
  }

  // ---- A and B by blocks of 16 x 16 tokens; a lane gets row r16, columns 4 g ..
  constexpr int BW = (10 + W - 1) / W;
  f32x4 blk[BW][HEADS];
#pragma unroll
  for (int m = 0; m < BW; ++m) {
    const int idx = wave + W * m;
    if (idx >= 10) continue;
    int I, J;
    block_place(idx, I, J);
    const T *ki = ks + (16 * I + r16) * KS + 8 * g, *kj = ks + (16 * J + r16) * KS + 8 * g, *qi = qs + (16 * I + r16) * KS + 8 * g;
    f32x4 kk = {0.f, 0.f, 0.f, 0.f}, qk = kk;
#pragma unroll
    for (int s = 0; s < NK; ++s) {
      const u32x4 right = *(const u32x4 *)(kj + 32 * s);
      kk = mfma16x16x32<B16>(right, *(const u32x4 *)(ki + 32 * s), kk);
      qk = mfma16x16x32<B16>(right, *(const u32x4 *)(qi + 32 * s), qk);
    }
    const int i = 16 * I + r16, j0 = 16 * J + 4 * g;
#pragma unroll
    for (int h = 0; h < HEADS; ++h) {
      const float *r = rss + h * L;
      const float ri = r[i], fi = -bts[h * L + i] * fk[i], gi = fq[i];
      f32x4 A, B;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float f = fk[j0 + e] * __builtin_amdgcn_exp2f(j0 + e <= i ? ri - r[j0 + e] : 0.f);
        A[e] = j0 + e < i ? kk[e] * (fi * f) : 0.f;
        B[e] = j0 + e <= i ? qk[e] * (gi * f) : 0.f;
      }
      blk[m][h] = A;   // (the negative)
      u32x2 hi, lo;
      split4(B, hi, lo);
      u32x2 *dst = (u32x2 *)(ws + (h - of) * kScalarTotal * 1024 + (kB + triangle(I, J >> 1) * 2) * 1024 + lane * 16) + (J & 1);
      dst[0] = hi;
      dst[128] = lo;
      if (I == J && (I & 1) == 0) dst[1] = dst[129] = u32x2{0u, 0u};   // the columns behind, in the same step of 32
    }
  }
  __syncthreads();   // k and q are done with
#pragma unroll
  for (int m = 0; m < BW; ++m) {
    const int idx = wave + W * m;
    if (idx >= 10) continue;
    int I, J;
    block_place(idx, I, J);
#pragma unroll
    for (int h = 0; h < HEADS; ++h)
      *(f32x4 *)((float *)(h ? (char *)ks : (char *)qs) + (16 * I + r16) * TS + 16 * J + 4 * g) = blk[m][h];
  }
  __syncthreads();
  solve_chunk(ts, bt, wave & 3, lane);
  for (int m = wave & 3; m < kTriangle; m += 4) {
    u32x4 hi, lo;
    solution_operand(ts, m, lane, hi, lo);
    u32x4 *dst = (u32x4 *)(ws + m * 2 * 1024) + lane;
    dst[0] = hi, dst[64] = lo;
  }
}

// Workgroup = W waves = W tiles of 16 columns of one head of one sequence; a wave keeps S of its columns in accumulators, whose rows are
// dealt so that tiles 2 s and 2 s + 1 together hold n = 32 s + 8 g .. + 7 in lane group g: operands of the next product as they are.  o is
// computed transposed (columns by tokens), so that a lane holds four columns of a token; the rows of v land in LDS like those of k and q and are
// read transposed, and o leaves by way of their place as whole lines.
// Bound by the chain of a chunk (132 products and some 500 vector instructions of a wave, each part waiting for the one before) and by the way of its
// 75 KB through the memory pipeline.  16 heads of 128 x 128, 16 sequences of 745 .. 1490 tokens: 198 us with four waves of two tiles, v and o by
// elements; 158 with eight waves of one tile, two on a SIMD, that fill each other's gaps, and v by LDS; 144 with transfers asked for between the
// products (all at once they held a wave up for 3000 of 12000 cycles) and k, q on one XCD; 135 with o by lines (by 32 bytes its stores took 30 us).
// Where heads and sequences do not fill the chip, workgroups of four waves leave no CU idle.
// NORM (the workgroup has all of a head's columns): the rows leave normed and gated.  A row of the head lies on 2 W adjacent lanes when it is stored, as in
// head_norm_gate_kernel, whose rounding points and order of the sum these are; the gate's pieces come with the chunk.  Bound by the same
// chain, of which this is vector arithmetic: the walk above 140 -> 174 us under the profiler, where a launch behind it took 53 and a pass over o; the layer 271 -> 245.  Half of
// the waves later than the others, so that one of two on a SIMD multiplies meanwhile: 267.
template <int NK, int W, bool NORM>
__global__ void __launch_bounds__(W * 64, 1) delta_scalar_walk_kernel(DeltaPrep q) {
  typedef elem<B16>::T T;
  constexpr int N = NK * 32, ROWS = 4 * NK, VF = 2 * W;   // fragments of 1 KiB: k, q; v
  constexpr int AT_V = 2 * ROWS, AT = AT_V + VF, STAGE = (AT + kScalarTotal) * 1024, PER = (kScalarTotal + W - 1) / W;
  const MvDeltaArgs &p = q.a;
  extern __shared__ __attribute__((aligned(16))) char smem[];   // 2 stages of k [4][NK] | q [4][NK] | v [64][W * 16] | T | B | factors
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4;
  // (workgroups are dealt to the 8 XCDs in turn: each gets a run of columns and heads, which share k and q)
  const int wide = gridDim.x, all = wide * p.heads;
  int at_head = blockIdx.y * wide + blockIdx.x;
  if (!(all & 7)) at_head = (at_head & 7) * (all >> 3) + (at_head >> 3);
  const int head = at_head / wide, seq = blockIdx.z, tiles = p.p / 16, tile0 = (at_head - head * wide) * W, grp = head / (p.heads / p.groups);
  const int q0 = p.cu_q[seq], len = p.cu_q[seq + 1] - q0;
  if (len <= 0) return;
  const int before = p.cu_k[seq + 1] - p.cu_k[seq] - len, slot = p.state_slots[seq];
  const bool keep = slot >= 0 && slot < p.slots;
  const int64_t size = (int64_t)p.heads * p.n * p.p;
  const int64_t stride = (int64_t)p.heads * kScalarTotal * 1024;
  const char *ws = q.ws + ((int64_t)(q0 / L + seq) * p.heads + head) * kScalarTotal * 1024 + lane * 16;
  const T *x = (const T *)p.x + (int64_t)q0 * p.x_stride;

  const bool live = tile0 + wave < tiles;
  const int col = min(tile0 + wave, tiles - 1) * 16;
  auto state_at = [&](int half, int i, int e) {
    const int n = (i >> 1) * 32 + g * 8 + (i & 1) * 4 + e;
    return p.state + half * p.slots * size + (int64_t)(keep ? slot : 0) * size + ((int64_t)head * p.n + n) * p.p + col + r16;
  };
  f32x4 st[2 * NK];
#pragma unroll
  for (int i = 0; i < 2 * NK; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) st[i][e] = keep && before > 0 ? *state_at(before & 1, i, e) : 0.f;

  auto transfer = [&](const void *from, char *to) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)from, (__attribute__((address_space(3))) void *)to, 16, 0, 0);
  };
  // Where this lane's pieces of 16 bytes come from: rows of k and q of one token tile (of half its channels, with eight waves), two runs of rows of v
  // (whose pieces lie in an order that spreads eight rows over the banks), its share of the rest.  Rows behind the end: the last row again, with
  // factors 0.
  constexpr int VP = 2 * W, VR = 64 / VP;   // pieces of a row of v, rows of a fragment
  auto v_swizzle = [](int row) { return (row << 1) & (VP - 1); };
  constexpr int KQ = (NK + W / 4 - 1) / (W / 4) * 2, ALL = KQ + 2 + PER;   // transfers of a wave and chunk
  auto fetch = [&](auto I, int c) __attribute__((always_inline)) {
    constexpr int n = decltype(I)::value;
    char *to = smem + (c & 1) * STAGE;
    if constexpr (n < KQ) {
      const int it = wave & 3, s = n / 2 * (W / 4) + (wave >> 2);
      const T *row = x + (int64_t)min(c * L + 16 * it + (lane >> 2), len - 1) * p.x_stride + grp * N + row_chunk(lane) * 8;
      if (NK % (W / 4) == 0 || s < NK) transfer(row + (n % 2 ? p.q_off : p.k_off) + 32 * s, to + (n % 2 * ROWS + it * NK + s) * 1024);
    } else if constexpr (n < KQ + 2) {
      const int f = 2 * wave + n - KQ, r = f * VR + lane / VP, piece = (lane % VP) ^ v_swizzle(r);
      const T *from = x + (int64_t)min(c * L + r, len - 1) * p.x_stride + head * p.p + min(tile0 * 16 + piece * 8, p.p - 8);
      transfer(from, to + (AT_V + f) * 1024);
    } else {
      const int f = min((n - KQ - 2) * W + wave, kScalarTotal - 1);
      transfer(ws + c * stride + f * 1024, to + (AT + f) * 1024);
    }
  };
  // Results take the place of the wave's columns of v in LDS; at the next chunk a wave takes the rows from there that it brings v of, whole lines
  // of them, and stores them.
  u32x4 done[2], gate[2] = {}, norm_w[2];   // (gate: of the chunk's rows, on their way with it)
  const bool padded = p.p_true < W * 16;
  auto col_of = [&](int i) { return ((lane % VP) ^ v_swizzle((2 * wave + i) * VR + lane / VP)) * 8; };   // (the head's first column is the workgroup's)
  if constexpr (NORM) {
#pragma unroll
    for (int i = 0; i < 2; ++i) norm_w[i] = *(const u32x4 *)((const T *)p.norm_w + min(col_of(i), p.p - 8));
  }
  auto ask_gate = [&](int c, int i) __attribute__((always_inline)) {
    const int t = min(c * L + (2 * wave + i) * VR + lane / VP, len - 1);
    gate[i] = *(const u32x4 *)((const T *)p.gate + (int64_t)(q0 + t) * p.gate_stride + head * p.p + min(col_of(i), p.p - 8));
  };
  auto norm_gate = [&](int i) __attribute__((always_inline)) {   // done[i] becomes what norm and gate make of it
    float f[8], z[8], w[8], ss = 0.f;
    unpack8<B16>(done[i], f);
    unpack8<B16>(gate[i], z);
    unpack8<B16>(norm_w[i], w);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (padded && col_of(i) + j >= p.p_true) f[j] = 0.f;
      ss = fmaf(f[j], f[j], ss);
    }
    const float rs = head_rms(lanes_sum<VP>(ss), p.p_true, p.eps, p.out_scale);
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = f[j] * rs * w[j] * gate_16(z[j], p.gate_kind);
    done[i] = pack8<B16>(f);
  };
  const bool pieces = !(((uintptr_t)p.out & 15) | (p.out_stride & 7));   // (rows of the output may stand anywhere)
  auto store = [&](int c, int i) __attribute__((always_inline)) {
    const int r = (2 * wave + i) * VR + lane / VP, t = c * L + r, at = tile0 * 16 + ((lane % VP) ^ v_swizzle(r)) * 8;
    if (t >= len || at >= p.p) return;
    T *to = (T *)p.out + (int64_t)(q0 + t) * p.out_stride + head * p.p + at;
    if (pieces) {
      *(u32x4 *)to = done[i];
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) to[e] = (T)(done[i][e >> 1] >> (e & 1) * 16);
    }
  };
  // What a chunk's transfers and stores cost is their way through the memory pipeline, which a wave that asks for all of them at once waits out: they
  // are asked for a few at a time, between its products.
  constexpr int POINTS = NK + 1;
  auto between = [&](auto I, int c, int chunks) __attribute__((always_inline)) {
    constexpr int n = decltype(I)::value, lo = ALL * n / POINTS, hi = ALL * (n + 1) / POINTS;
    if constexpr (n == 0) lds_wait<8>(done[0], done[1]);   // (read ahead of the rows; the transfers of v come behind)
    if (c + 1 < chunks) static_for<hi - lo>([&](auto J) { fetch(std::integral_constant<int, lo + decltype(J)::value>{}, c + 1); });
    if constexpr (n < 2) {
      if (c > 0) {
        if constexpr (NORM) norm_gate(n);
        store(c - 1, n);
      }
      if constexpr (NORM) ask_gate(c, n);
    }
  };
  const uint32_t lds = lds_address(smem);
  const int chunks = (len + L - 1) / L;
  static_for<ALL>([&](auto I) { fetch(I, 0); });
  for (int c = 0; c < chunks; ++c) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    lds_barrier();   // this chunk has landed; every wave is done with the one before
    // (the compiler's own wait for the gate belongs here, where nothing is under way: behind, it would take in the next chunk's transfers)
    if constexpr (NORM) asm volatile("" : "+v"(gate[0]), "+v"(gate[1]));
    const uint32_t at = lds + (c & 1) * STAGE, rows = at + row_place(r16, g) * 16, rest_at = at + AT * 1024;
    const uint32_t fl = rest_at + lane * 16, ff = rest_at + kFactors * 1024 + g * 16;
    const uint32_t tr = at + row_place(4 * g + (r16 >> 2), r16 & 3) * 16;
    const int vrow = 4 * g + (r16 >> 2);   // (rows 16 apart have the same order)
    const uint32_t vt = at + AT_V * 1024 + vrow * W * 32 + ((2 * wave + ((r16 & 3) >> 1)) ^ v_swizzle(vrow)) * 16 + (r16 & 1) * 8;
    // ---- k S (tokens by columns) and q S (columns by tokens); what comes out of LDS is asked for one step ahead, here and below
    f32x4 ksum[4], o[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) ksum[it] = o[it] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 fk[2][4], fq[2][4], raw[2][4];
    u32x2 v[4];
    float to_o[4], last;
    auto read_rows = [&](auto S) __attribute__((always_inline)) {
      constexpr int s = decltype(S)::value;
      static_for<4>([&](auto I) {
        constexpr int it = decltype(I)::value;
        lds_read128<(it * NK + s) * 1024>(fk[s & 1][it], rows);
        lds_read128<(ROWS + it * NK + s) * 1024>(fq[s & 1][it], rows);
      });
    };
    const uint32_t results = lds + ((c + 1) & 1) * STAGE + (AT_V + 2 * wave) * 1024 + lane * 16;
    lds_read128<0>(done[0], results);
    lds_read128<1024>(done[1], results);
    read_rows(std::integral_constant<int, 0>{});
    static_for<NK>([&](auto S) {
      constexpr int s = decltype(S)::value;
      u32x4 sh, sl;
      if constexpr (s + 1 < NK) {
        read_rows(std::integral_constant<int, s + 1>{});
      } else {
        static_for<4>([&](auto I) {
          constexpr int it = decltype(I)::value;
          lds_read64_tr<it * 16 * W * 32>(v[it], vt);
          lds_read128<it * 64>(raw[0][it], ff);
        });
      }
      split44(st[2 * s], st[2 * s + 1], sh, sl);
      static_for<4>([&](auto I) {
        constexpr int it = decltype(I)::value;
        lds_wait<8>(fk[s & 1][it], fq[s & 1][it]);
      });
#pragma unroll
      for (int part = 0; part < 2; ++part)
#pragma unroll
        for (int it = 0; it < 4; ++it) {
          ksum[it] = mfma16x16x32<B16>(fk[s & 1][it], part ? sl : sh, ksum[it]);
          o[it] = mfma16x16x32<B16>(part ? sl : sh, fq[s & 1][it], o[it]);
        }
      between(S, c, chunks);
    });
    // ---- R, U = T R
    u32x4 ft[2][kTriangle][2];   // T, B
    auto read_triangle = [&](auto B) __attribute__((always_inline)) {
      constexpr int b = decltype(B)::value;
      static_for<kTriangle>([&](auto M) {
        constexpr int m = decltype(M)::value;
        lds_read128<b * kB * 1024 + m * 2048>(ft[b][m][0], fl);
        lds_read128<b * kB * 1024 + m * 2048 + 1024>(ft[b][m][1], fl);
      });
    };
    read_triangle(std::integral_constant<int, 0>{});
    static_for<4>([&](auto I) {
      constexpr int it = decltype(I)::value;
      lds_wait<2 * kTriangle>(raw[0][it]);
      lds_wait<2 * kTriangle>(v[it]);
    });
    u32x4 uh[2], ul[2];
    f32x4 rest[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const f32x4 f = __builtin_bit_cast(f32x4, raw[0][it]) * ksum[it];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        rest[it][2 * e] = u2f(v[it][e] << 16) - f[2 * e];
        rest[it][2 * e + 1] = u2f(v[it][e] & 0xffff0000u) - f[2 * e + 1];
      }
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) split44(rest[2 * s], rest[2 * s + 1], uh[s], ul[s]);
    f32x4 u[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) u[it] = f32x4{0.f, 0.f, 0.f, 0.f};
    static_for<kTriangle>([&](auto M) { lds_wait<0>(ft[0][decltype(M)::value][0], ft[0][decltype(M)::value][1]); });
    static_for<4>([&](auto I) {
      constexpr int it = decltype(I)::value;
      lds_read32<kFactors * 1024 + 256 + it * 64>(to_o[it], rest_at + r16 * 4);
    });
    read_triangle(std::integral_constant<int, 1>{});
#pragma unroll
    for (int part = 0; part < 3; ++part)
      static_for<4>([&](auto I) {
        constexpr int it = decltype(I)::value;
        static_for<it / 2 + 1>([&](auto S) {
          constexpr int s = decltype(S)::value;
          u[it] = mfma16x16x32<B16>(ft[0][triangle(it, s)][part == 2], part == 1 ? ul[s] : uh[s], u[it]);
        });
      });
    between(std::integral_constant<int, NK>{}, c, chunks);
    // ---- o += B U
    static_for<4>([&](auto I) {
      constexpr int it = decltype(I)::value;
      lds_wait<2 * kTriangle>(to_o[it]);
      o[it] *= to_o[it];
    });
#pragma unroll
    for (int s = 0; s < 2; ++s) split44(u[2 * s], u[2 * s + 1], uh[s], ul[s]);
    static_for<kTriangle>([&](auto M) { lds_wait<0>(ft[1][decltype(M)::value][0], ft[1][decltype(M)::value][1]); });
    // ---- k transposed: row r16 of a state tile, tokens 16 (e >> 2) + 4 g + (e & 3) of a step of 32
    u32x2 kt[2][2][2][2];   // [which][state tile][step of 32 tokens][its half]
    auto read_pair = [&](auto P) __attribute__((always_inline)) {
      constexpr int pair = decltype(P)::value;
      static_for<2>([&](auto D) {
        constexpr int d = decltype(D)::value;
        static_for<4>([&](auto I) {
          constexpr int it = decltype(I)::value;
          lds_read64_tr<(it * NK + pair) * 1024 + d * 8>(kt[pair & 1][d][it >> 1][it & 1], tr);
        });
      });
    };
    static_for<4>([&](auto I) {
      constexpr int it = decltype(I)::value;
      lds_read128<it * 64 + 512>(raw[1][it], ff);
    });
    lds_read32<kFactors * 1024 + 768>(last, rest_at);
    read_pair(std::integral_constant<int, 0>{});
#pragma unroll
    for (int part = 0; part < 3; ++part)
      static_for<4>([&](auto I) {
        constexpr int it = decltype(I)::value;
        static_for<it / 2 + 1>([&](auto S) {
          constexpr int s = decltype(S)::value;
          o[it] = mfma16x16x32<B16>(part == 1 ? ul[s] : uh[s], ft[1][triangle(it, s)][part == 2], o[it]);
        });
      });
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int row = 16 * it + r16;
      *(u32x2 *)(smem + (c & 1) * STAGE + AT_V * 1024 + row * W * 32 + ((2 * wave + (g >> 1)) ^ v_swizzle(row)) * 16 + (g & 1) * 8) = pack_quad<B16>(o[it]);
    }
    // ---- S <- decay S + k^T (e^{r_last - r} f u)
    static_for<4>([&](auto I) {
      constexpr int it = decltype(I)::value;
      lds_wait<8>(raw[1][it]);
      u[it] *= __builtin_bit_cast(f32x4, raw[1][it]);
    });
    lds_wait<8>(last);
#pragma unroll
    for (int s = 0; s < 2; ++s) split44(u[2 * s], u[2 * s + 1], uh[s], ul[s]);
#pragma unroll
    for (int i = 0; i < 2 * NK; ++i) st[i] *= last;
    static_for<NK>([&](auto P) {
      constexpr int pair = decltype(P)::value;
      if constexpr (pair + 1 < NK) read_pair(std::integral_constant<int, pair + 1>{});
      static_for<2>([&](auto D) {
        constexpr int d = decltype(D)::value;
        lds_wait<(pair + 1 < NK ? 8 : 0)>(kt[pair & 1][d][0][0], kt[pair & 1][d][0][1]);
        lds_wait<(pair + 1 < NK ? 8 : 0)>(kt[pair & 1][d][1][0], kt[pair & 1][d][1][1]);
      });
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int part = 0; part < 2; ++part)
#pragma unroll
          for (int d = 0; d < 2; ++d) {
            const u32x2 &lo = kt[pair & 1][d][s][0], &hi = kt[pair & 1][d][s][1];
            st[2 * pair + d] = mfma16x16x32<B16>(u32x4{lo[0], lo[1], hi[0], hi[1]}, part ? ul[s] : uh[s], st[2 * pair + d]);
          }
    });
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  lds_barrier();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    done[i] = *(const u32x4 *)(smem + ((chunks - 1) & 1) * STAGE + (AT_V + 2 * wave + i) * 1024 + lane * 16);
    if constexpr (NORM) norm_gate(i);
    store(chunks - 1, i);
  }
  if (keep && live) {
#pragma unroll
    for (int i = 0; i < 2 * NK; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) *state_at((before + len) & 1, i, e) = st[i][e];
  }
}

template <int NK, int W>
int launch_walk(const DeltaPrep &q, int slices, int lds, bool *normed, hipStream_t stream) {
  const dim3 grid(slices, q.a.heads, q.a.n_seqs), block(W * 64);
  // Norm and gate in the walk lengthen the chain of the longest sequence, by some 1.2 us a chunk with eight waves and 0.5 (64 key channels) to 0.7 with four; a launch
  // behind it takes 2.5 us and the time of its rows, 4.6 TB/s.  us, in the walk and behind: 16 heads over 8 of 128 x 128, 40 sequences of up to 600 tokens 192 and 215; of 64 x 64,
  // 16 of up to 1490 116 and 124, 3 of up to 600 44 and 41, 8 of up to 3000 168 and 162, over 16 191 and 206; 3 heads of 32 x 32, 40 of up to 600 45 and 42.
  const double chunks = (q.a.max_q + L - 1) / L, in_chain = chunks * (W == 8 ? 1.2 : 0.65), behind = 2.5 + (double)q.a.total_q * q.a.heads * q.a.p * 6 / 4.6e6;
  const bool in_walk = normed && slices == 1 && (*normed || in_chain <= behind);
  if (normed) *normed = in_walk;
  if (in_walk) {
    if (int rc = mv_allow_lds<delta_scalar_walk_kernel<NK, W, true>>()) return rc;
    hipLaunchKernelGGL((delta_scalar_walk_kernel<NK, W, true>), grid, block, lds, stream, q);
  } else {
    if (int rc = mv_allow_lds<delta_scalar_walk_kernel<NK, W, false>>()) return rc;
    hipLaunchKernelGGL((delta_scalar_walk_kernel<NK, W, false>), grid, block, lds, stream, q);
  }
  MV_LAUNCH_CHECK();
  return MV_OK;
}

template <int NK>
int launch(const DeltaPrep &q, bool *normed, hipStream_t stream) {
  const MvDeltaArgs &a = q.a;
  const unsigned slots = (unsigned)chunk_slots(a.n_seqs, a.total_q);
  const int of_group = a.heads / a.groups;
  if (q.raw && of_group == 2) hipLaunchKernelGGL((delta_scalar_prepare_kernel<NK, 2, true>), dim3(slots, a.heads / 2), dim3(512), 0, stream, q);
  else if (q.raw) hipLaunchKernelGGL((delta_scalar_prepare_kernel<NK, 1, true>), dim3(slots, a.heads), dim3(256), 0, stream, q);
  else if (of_group % 2 == 0) hipLaunchKernelGGL((delta_scalar_prepare_kernel<NK, 2, false>), dim3(slots, a.heads / 2), dim3(512), 0, stream, q);
  else hipLaunchKernelGGL((delta_scalar_prepare_kernel<NK, 1, false>), dim3(slots, a.heads), dim3(256), 0, stream, q);
  MV_LAUNCH_CHECK();
  // Eight waves where workgroups of four would be more than the CUs, of which each holds one, and LDS holds their chunk (up to 128 channels: at
  // 160 four waves of one tile it is, 16 heads and 16 sequences of 1000 tokens 201 us, where four waves of two tiles took 211)
  const int tiles = a.p / 16, wide = (tiles + 7) / 8, narrow = (tiles + 3) / 4;
  constexpr auto lds = [](int waves) { return 2 * (8 * NK + 2 * waves + kScalarTotal) * 1024; };
  if constexpr (lds(8) <= 160 * 1024) {
    if (tiles > 4 && (int64_t)narrow * a.heads * a.n_seqs > 256) return launch_walk<NK, 8>(q, wide, lds(8), normed, stream);
  }
  return launch_walk<NK, 4>(q, narrow, lds(4), normed, stream);
}

}  // namespace

// (arguments checked by mv_delta_chunk_launch, whose workspace is larger)
int mv_delta_scalar_launch(const MvDeltaArgs &a, const void *raw, int64_t raw_stride, bool *normed, hipStream_t stream) {
  const DeltaPrep q{a, (char *)a.workspace, raw, raw_stride};
  switch (a.n / 32) {
    case 1: return launch<1>(q, normed, stream);
    case 2: return launch<2>(q, normed, stream);
    case 3: return launch<3>(q, normed, stream);
    case 4: return launch<4>(q, normed, stream);
    case 5: return launch<5>(q, normed, stream);
  }
  return MV_E_SHAPE;
}
