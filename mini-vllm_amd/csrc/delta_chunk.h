// Shared by the chunked forms of the gated delta rule (K16): delta_chunk.hip, delta_scalar.hip.
#pragma once
#include "delta.h"

namespace {

constexpr int L = 64;              // tokens per chunk

typedef bf16_tag B16;

__device__ __forceinline__ void split8(const float (&f)[8], u32x4 &hi, u32x4 &lo) {
  float rest[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    hi[i] = pack_pair<B16>(f[2 * i], f[2 * i + 1]);
    rest[2 * i] = f[2 * i] - u2f(hi[i] << 16);
    rest[2 * i + 1] = f[2 * i + 1] - u2f(hi[i] & 0xffff0000u);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) lo[i] = pack_pair<B16>(rest[2 * i], rest[2 * i + 1]);
}
__device__ __forceinline__ void split44(const f32x4 &a, const f32x4 &b, u32x4 &hi, u32x4 &lo) {
  const float f[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  split8(f, hi, lo);
}
__device__ __forceinline__ f32x4 mfma3(const u32x4 &ah, const u32x4 &al, const u32x4 &bh, const u32x4 &bl, f32x4 c) {
  c = mfma16x16x32<B16>(ah, bh, c);
  c = mfma16x16x32<B16>(ah, bl, c);
  return mfma16x16x32<B16>(al, bh, c);
}
// softplus in hardware exponential and logarithm: an absolute error of about 1e-7
__device__ __forceinline__ float softplus_fast(float z) {
  return fmaxf(z, 0.f) + 0.6931471805599453f * __builtin_amdgcn_logf(1.f + __builtin_amdgcn_exp2f(-1.4426950408889634f * fabsf(z)));
}

struct DeltaPrep {
  MvDeltaArgs a;
  char *ws;
  const void *raw;      // channels ahead of the convolution, or NULL: a.x is there already
  int64_t raw_stride;
};

// chunk slot -> sequence (its slots start at cu_q / L + its number)
__device__ __forceinline__ int chunk_sequence(const MvDeltaArgs &p, int slot) {
  int seq = 0;
  for (int hi = p.n_seqs; hi - seq > 1;) {
    const int mid = (seq + hi) >> 1;
    if (p.cu_q[mid] / L + mid <= slot) seq = mid;
    else hi = mid;
  }
  return seq;
}
constexpr int kChunkTaps = 4;
// The causal convolution of kChunkTaps taps and silu of causal_conv_kernel (the same sums) for a chunk's channels of a group, THREADS threads, four channels and
// eight tokens a thread and turn: k and q of group `grp` (N channels each), `values` of v from `first` on.  put(0: k, 1: q, 2: v; row; place among those channels;
// channel; results, zeros behind the end): every row of k and q, with ALL of v too.  What is kept of the inputs is written along with a sequence's first rows.
template <typename Tag, int N, int THREADS, bool ALL, typename Put>
__device__ __forceinline__ void conv_chunk(const DeltaPrep &q, int seq, int q0, int len, int t0, int nt, int grp, int first, int values, int tid, Put put) {
  typedef uint16_t T;
  constexpr int TAPS = kChunkTaps, ROWS = 8, back = TAPS - 1;
  const MvDeltaArgs &p = q.a;
  const int before = p.cu_k[seq + 1] - p.cu_k[seq] - len, slot = p.state_slots[seq];
  const bool keep = slot >= 0 && slot < p.slots;
  const int64_t half = p.slots * back * p.channels;
  const T *conv_w = (const T *)p.conv_w, *from = (const T *)q.raw + (int64_t)q0 * q.raw_stride;
  const T *old_state = (const T *)p.conv_state + (before & 1) * half + (int64_t)(keep ? slot : 0) * back * p.channels;
  const int pieces = (2 * N + values) / 4;   // of a token
  const auto unpack4 = [](const u32x2 &v, float (&f)[4]) {
    float all[8];
    unpack8<Tag>(u32x4{v[0], v[1], 0u, 0u}, all);
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = all[i];
  };
  for (int item = tid; item < pieces * (L / ROWS); item += THREADS) {
    const int piece = item % pieces, tr = item / pieces * ROWS, which = min(piece / (N / 4), 2), at = (piece - which * (N / 4)) * 4;
    const int c = which == 0 ? p.k_off + grp * N + at : which == 1 ? p.q_off + grp * N + at : first + at;
    auto input = [&](int t) {   // input `t` of the step (t < 0: of the steps before it)
      if (t >= 0) return *(const u32x2 *)(from + (int64_t)min(t, len - 1) * q.raw_stride + c);
      if (before > 0 && keep) return *(const u32x2 *)(old_state + (int64_t)(back + t) * p.channels + c);
      return u32x2{0u, 0u};
    };
    float w[TAPS][4], win[TAPS][4];
    if (!ALL && tr >= nt && which > 1) continue;
    u32x2 raw[back], rows[ROWS];
#pragma unroll
    for (int i = 0; i < back; ++i) raw[i] = input(t0 + tr + i - back);
#pragma unroll
    for (int u = 0; u < ROWS; ++u) rows[u] = input(t0 + tr + u);
#pragma unroll
    for (int i = 0; i < TAPS; ++i) unpack4(*(const u32x2 *)(conv_w + (int64_t)i * p.channels + c), w[i]);
#pragma unroll
    for (int i = 0; i < back; ++i) unpack4(raw[i], win[i + 1]);   // shifted down below
    if (t0 + tr == 0 && keep) {   // the only thread that reads the old state here writes the new one, behind its reads
      u32x2 last[back];
#pragma unroll
      for (int j = 0; j < back; ++j) last[j] = input(len - back + j);
      T *ns = (T *)p.conv_state + ((before + len) & 1) * half + (int64_t)slot * back * p.channels + c;
#pragma unroll
      for (int j = 0; j < back; ++j) *(u32x2 *)(ns + (int64_t)j * p.channels) = last[j];
    }
#pragma unroll
    for (int u = 0; u < ROWS; ++u) {
#pragma unroll
      for (int i = 0; i < back; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) win[i][j] = win[i + 1][j];
      unpack4(rows[u], win[back]);
      float o[8] = {};   // (four of them: packed as causal_conv_kernel packs eight)
#pragma unroll
      for (int i = 0; i < TAPS; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = fmaf(win[i][j], w[i][j], o[j]);
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = silu_of<Tag>(o[j]);
      const u32x4 done = pack8<Tag>(o);
      put(which, tr + u, at, c, tr + u < nt ? u32x2{done[0], done[1]} : u32x2{0u, 0u});
    }
  }
}

inline int64_t chunk_slots(int n_seqs, int total_q) { return (int64_t)total_q / L + n_seqs; }

// the ten blocks of 16 x 16 tokens on and below the diagonal, dealt over the waves
__device__ __forceinline__ void block_place(int idx, int &I, int &J) {
  I = idx < 4 ? 3 : idx < 7 ? 2 : idx < 9 ? 1 : 0, J = idx < 4 ? 3 - idx : idx < 7 ? 6 - idx : idx < 9 ? 8 - idx : 0;
}

// an accumulator as half of an operand, high parts and rests
__device__ __forceinline__ void split4(const f32x4 &f, u32x2 &hi, u32x2 &lo) {
  hi = pack_quad<B16>(f);
  f32x4 rest;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    rest[2 * e] = f[2 * e] - u2f(hi[e] << 16);
    rest[2 * e + 1] = f[2 * e + 1] - u2f(hi[e] & 0xffff0000u);
  }
  lo = pack_quad<B16>(rest);
}

constexpr int TS = L + 4;   // row stride of A and T in LDS
// operands of a lower triangular matrix of L x L tokens: (token tile, step of 32 tokens) 0 0, 1 0, 2 0, 2 1, 3 0, 3 1
constexpr int kTriangle = 6;
__host__ __device__ constexpr int triangle(int it, int s) { return it < 2 ? it : 2 * it - 2 + s; }

// T = (1 + A)^-1 diag(beta), in place of -A in LDS (-A is there, behind a barrier; so is T afterwards), by the first four waves.  T's entries are
// at most 1, since no factor 1 - beta k k^T of the recurrence lengthens a vector.
__device__ __forceinline__ void solve_chunk(float *ts, const float *bt, int wave, int lane) {
  const int r16 = lane & 15, g = lane >> 4;
  // A wave inverts a diagonal block, a column in each of 16 lanes, into one of the blocks above the diagonal, which nothing uses ..
  auto inverse = [&](int I) { return ts + (I < 3 ? 16 * (I + 1) : 16 * TS + 32); };
  if (wave < 4 && lane < 16) {
    const float *d = ts + 16 * wave * TS + 16 * wave;
    float *to = inverse(wave), x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float a = i == r16 ? 1.f : 0.f, b = 0.f;
#pragma unroll
      for (int j = 0; j < i; j += 4) {   // (zeros from column i on)
        const f32x4 t = *(const f32x4 *)(d + i * TS + j);
        a = fmaf(t[0], x[j], a);
        if (j + 1 < i) b = fmaf(t[1], x[j + 1], b);
        if (j + 2 < i) a = fmaf(t[2], x[j + 2], a);
        if (j + 3 < i) b = fmaf(t[3], x[j + 3], b);
      }
      x[i] = a + b;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) to[i * TS + r16] = x[i];
  }
  __syncthreads();
  // .. and then a wave a column of blocks, from the diagonal down: T_IJ = T_II sum_{J <= K < I} (-A_IK) T_KJ.  Accumulators are the
  // right operand of the next product, whose keys are 4 g + step.
  f32x4 t[4];
  if (wave < 4) {
    auto product = [&](const float *block, const f32x4 &right, f32x4 acc) {
      const f32x4 left = *(const f32x4 *)(block + r16 * TS + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(left[e], right[e], acc, 0, 0, 0);
      return acc;
    };
#pragma unroll
    for (int I = 0; I < 4; ++I) {
      t[I] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (I < wave) continue;
      if (I == wave) {
#pragma unroll
        for (int e = 0; e < 4; ++e) t[I][e] = inverse(I)[(4 * g + e) * TS + r16];
        continue;
      }
      f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int K = 0; K < I; ++K)
        if (K >= wave) sum = product(ts + 16 * I * TS + 16 * K, t[K], sum);
      t[I] = product(inverse(I), sum, t[I]);
    }
  }
  __syncthreads();   // every wave has read A
  if (wave < 4) {
    const float beta = bt[16 * wave + r16];
#pragma unroll
    for (int I = 0; I < 4; ++I)
      if (I >= wave) {
#pragma unroll
        for (int e = 0; e < 4; ++e) ts[(16 * I + 4 * g + e) * TS + 16 * wave + r16] = t[I][e] * beta;
      }
  }
  __syncthreads();
}

// rows of T as an operand of either side: row r16 of a token tile, tokens 16 (e >> 2) + 4 g + (e & 3) of a step of 32
__device__ __forceinline__ void solution_operand(const float *ts, int m, int lane, u32x4 &hi, u32x4 &lo) {
  const int it = m < 2 ? m : 2 + (m - 2) / 2, s = m < 2 ? 0 : m & 1;
  const float *row = ts + (16 * it + (lane & 15)) * TS + 32 * s + 4 * (lane >> 4);
  const f32x4 a = *(const f32x4 *)row;
  f32x4 b = {0.f, 0.f, 0.f, 0.f};
  if (2 * s + 1 <= it) b = *(const f32x4 *)(row + 16);
  split44(a, b, hi, lo);
}

}  // namespace
