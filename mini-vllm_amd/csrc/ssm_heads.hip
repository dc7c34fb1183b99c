// K15 — the chunked recurrence of ssm_chunk.hip for heads of 64 columns that share b and c: four heads of a group to a workgroup, two waves each.
//
// There, a workgroup is a head, whose four waves of 16 columns each read all of b and c out of LDS: its vector instructions, its LDS reads and its products took
// turns, 3.1 us a chunk and head of a CU.  Here a wave has 32 columns, so that LDS reads are half as many, b and c are staged once for four heads (two stages,
// asked for a chunk ahead, without a trip through registers), and the vector unit makes the state's next parts while the matrix cores are at the ones before.  Per
// element below the diagonal tiles the weight is two products instead of an exponential.  2.2 us a chunk and head of a CU: a row's 12 chunks of four heads take the
// outputs' launch 99 .. 105 us, its start and end included, 16 500 cycles each (counters, at 2.0 GHz).  LDS reads (744 KB, at the 115 bytes a cycle that they reach) are 6500 of
// them, products 5700 (the matrix cores are busy for 34 % of the launch), vector instructions 6500; the two waves of a SIMD are in the same phase most of the time, so that these
// take turns in part.  A workgroup takes a CU's LDS, so that sequences as workgroups would leave half of the chip idle: the chunks of all sequences are dealt out evenly instead
// (Rows).  So a sequence is cut where those ahead of it say, and its last bits differ with its neighbours (results within a unit, kept states within 2^-16 of their norm), also at
// sizes where a head a workgroup would take whole sequences, the same bits in any call: without scratch memory that still holds.  64 heads of 64 x 128, 4 sequences of up to 3900
// tokens, convolution and norm included: 258 -> 222 us (states 56 -> 45, outputs 145 -> 105 under the profiler).  Tried: scores of a chunk made once for the four heads and
// weighted by each wave (LDS reads 464 KB, vector instructions by a fifth more), and a third barrier for weights made once: as slow; both token tiles of a wave's scores at once,
// two steps ahead: 6 % slower.
#include <algorithm>

#include "ssm.h"

namespace {

constexpr int L = 64;        // tokens per chunk
constexpr int HEADS = 4;     // of a workgroup, two waves (of 32 columns) each
constexpr int P = 64;

__device__ __forceinline__ u32x4 join(const u32x2 &a, const u32x2 &b) { return u32x4{a.x, a.y, b.x, b.y}; }
// two accumulators as one operand: high parts and remainders
template <typename Tag>
__device__ __forceinline__ void split44(const f32x4 &a, const f32x4 &b, u32x4 &hi, u32x4 &lo) {
  const u32x2 ha = pack_quad<Tag>(a), hb = pack_quad<Tag>(b);
  hi = join(ha, hb);
  float h[8];
  unpack8<Tag>(hi, h);
  lo = join(pack_quad<Tag>(f32x4{a[0] - h[0], a[1] - h[1], a[2] - h[2], a[3] - h[3]}),
            pack_quad<Tag>(f32x4{b[0] - h[4], b[1] - h[5], b[2] - h[6], b[3] - h[7]}));
}
__device__ __forceinline__ void exchange32(uint32_t &a, uint32_t &b) { asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b)); }
__device__ __forceinline__ void exchange16(uint32_t &a, uint32_t &b) { asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b)); }
template <int OFF>
__device__ __forceinline__ void lds_write32(uint32_t a, float v) {
  asm volatile("ds_write_b32 %0, %1 offset:%2" : : "v"(a), "v"(v), "i"(OFF) : "memory");
}
template <int OFF>
__device__ __forceinline__ void lds_write128(uint32_t a, const u32x4 &v) {
  asm volatile("ds_write_b128 %0, %1 offset:%2" : : "v"(a), "v"(v), "i"(OFF) : "memory");
}
template <int N>
__device__ __forceinline__ void vm_wait() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }
__device__ __forceinline__ void transfer(const void *from, char *to) {
  __builtin_amdgcn_global_load_lds((const MV_AS1 void *)from, (MV_AS3 void *)to, 16, 0, 0);
}

// The chunks of all sequences, one behind the other, are dealt to rows of workgroups in equal runs.  What a row's last sequence adds to the state where it goes on
// in the next row: states [row][heads][n * p] (in the order of a wave's registers), what it decays by [row][heads] (log2), what a sequence that begins in the row
// and goes on comes with, first [row][heads][n * p].
// The first launch begins with steps [chunk][heads][2][64]: of a chunk's tokens the log2 decay from its start on and the step size.
struct Rows {
  float *states, *decays, *first, *steps;
  int least;   // chunks of a row
};
enum { STATES, OUTPUTS };

// the ten tiles of scores on and below the diagonal as operands of 32 keys: 0 0, 1 0, 2 0, 2 1, 3 0, 3 1
__host__ __device__ constexpr int operand(int it, int s) { return it < 2 ? it : 2 * it - 2 + s; }

template <int NK, int MODE>
constexpr int lds_bytes() {
  constexpr int rows = L * NK * 64;   // of b, or c
  return MODE == STATES ? 2 * rows + 8 * 4096 + 8 * 256 : 4 * rows + 8 * 4096 + 8 * 1536 + HEADS * 12 * 1024;
}

template <typename Tag, int NK, int MODE>
__global__ void __launch_bounds__(512, MODE == STATES && NK == 2 ? 4 : 2) ssm_heads_kernel(MvSsmArgs p, Rows sg) {
  typedef typename elem<Tag>::T T;
  constexpr bool OUT = MODE != STATES;
  constexpr int N = NK * 32, RB = N * 2, ROWS = L * RB, BC = OUT ? 2 * ROWS : ROWS;   // LDS rows of b and c
  constexpr int STEP = OUT ? 1536 : 256, AT_X = 2 * BC, AT_S = AT_X + 8 * 4096, AT_W = AT_S + 8 * STEP;
  constexpr int S_R = 0, S_DT = 256, S_ALL = 512, S_E = 768, S_G = 1024, S_W = OUT ? 1280 : 0;
  extern __shared__ __attribute__((aligned(16))) char smem[];   // 2 stages of b | c; x of the waves; step sizes of the waves; weighted scores of the heads
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
  const int of = wave >> 1, half = wave & 1, head = blockIdx.x * HEADS + of;
  // ---- this row's chunks, [lo, hi) of all; the sequence they begin in, [start, end)
  int chunks = 0;
  for (int i = lane; i < p.n_seqs; i += 64) chunks += (p.cu_q[i + 1] - p.cu_q[i] + L - 1) / L;
#pragma unroll
  for (int o = 1; o < 64; o *= 2) chunks += __shfl_xor(chunks, o, 64);
  chunks = __builtin_amdgcn_readfirstlane(chunks);
  const int run = max((chunks + (int)gridDim.y - 1) / (int)gridDim.y, sg.least), lo = (int)blockIdx.y * run, hi = min(lo + run, chunks);
  if (lo >= hi) return;
  int seq = 0, start = 0, end = 0;
  auto find = [&](int chunk) __attribute__((always_inline)) {
    for (int base = 0, before = 0; base < p.n_seqs; base += 64) {
      const int own = base + lane < p.n_seqs ? (p.cu_q[base + lane + 1] - p.cu_q[base + lane] + L - 1) / L : 0;
      int upto = own;
#pragma unroll
      for (int o = 1; o < 64; o *= 2) {
        const int v = __shfl_up(upto, o, 64);
        if (lane >= o) upto += v;
      }
      upto += before;
      const uint64_t behind = __ballot(upto > chunk);
      if (behind) {
        const int at = __ffsll((unsigned long long)behind) - 1;
        seq = base + at, end = __builtin_amdgcn_readlane(upto, at), start = end - __builtin_amdgcn_readlane(own, at);
        return;
      }
      before = __builtin_amdgcn_readlane(upto, 63);
    }
  };
  auto go_on = [&]() {   // to the next sequence that has any tokens
    do {
      ++seq, start = end, end += (p.cu_q[seq + 1] - p.cu_q[seq] + L - 1) / L;
    } while (end == start);
  };
  find(lo);
  if constexpr (!OUT) {   // a wave a head of a chunk, a lane a token (behind the end: dt = 0, no decay)
    const int h = blockIdx.x * HEADS + (wave & 3);
    const float na2 = -expf(elem<Tag>::ld(((const T *)p.a_log)[h])) * 1.4426950408889634f, bias = elem<Tag>::ld(((const T *)p.dt_bias)[h]);
    for (int i = lo + (wave >> 2); i < hi; i += 2) {
      while (end <= i) go_on();
      const int q0 = p.cu_q[seq], len = p.cu_q[seq + 1] - q0, t = (i - start) * L + lane;
      const float raw = elem<Tag>::ld(((const T *)p.dt)[(int64_t)(q0 + min(t, len - 1)) * p.dt_stride + h]), step = t < len ? softplus_f32(raw + bias) : 0.f;
      float r = na2 * step;
#pragma unroll
      for (int o = 1; o < 64; o *= 2) {
        const float v = __shfl_up(r, o, 64);
        if (lane >= o) r += v;
      }
      float *to = sg.steps + ((int64_t)i * p.heads + h) * 2 * L + lane;
      to[0] = r, to[L] = step;
    }
    find(hi - 1);
    if (end <= hi) return;   // (nobody asks for its state)
    __syncthreads();
  }
  const int grp = head / (p.heads / p.groups);
  const int64_t size = (int64_t)p.heads * N * P, col = head * P + half * 32;
  float decayed = 0.f;   // (STATES) log2 decay of the chunks so far

  const T *x = nullptr;   // of the sequence's tokens in this row
  int len = 0;
  // ---- transfers to LDS, 1 KiB each.  Rows of b and c: pieces of 16 bytes in an order that spreads 16 rows, and four pieces of 8 rows, over the banks
  auto swizzle = [](int row) { return NK == 4 ? (row & 3) << 2 | ((row >> 2) & 3) : ((row >> 1) & 1) << 2 | ((row >> 2) & 3); };
  constexpr int PIECES = RB / 16, RUN = 64 / PIECES, EACH = L / RUN / 8;   // pieces of a row; rows of a transfer; transfers of a wave
  const int stride = (int)p.x_stride, bcol = p.b_off + grp * N, ccol = p.c_off + grp * N;
  auto token = [&](int t0) { return min(t0, len - 1); };   // (behind the end: any token)
  auto fetch_bc = [&](int t0) __attribute__((always_inline)) {
    char *to = smem + (t0 / L & 1) * BC;
#pragma unroll
    for (int k = 0; k < EACH; ++k) {
      const int f = wave * EACH + k, row = f * RUN + lane / PIECES, piece = (lane % PIECES) ^ swizzle(row);
      const int u = token(t0);
      const T *src = x + (int64_t)u * stride + (uint32_t)((min(u + row, len - 1) - u) * stride + piece * 8);
      transfer(src + bcol, to + f * 1024);
      if constexpr (OUT) transfer(src + ccol, to + ROWS + f * 1024);
    }
  };
  constexpr int BCS = OUT ? 2 * EACH : EACH;
  auto fetch_x = [&](int t0, int s) __attribute__((always_inline)) {   // 32 tokens of the wave's columns
#pragma unroll
    for (int k = 2 * s; k < 2 * s + 2; ++k) {
      const int row = 16 * k + (lane >> 2), piece = (lane & 3) ^ ((lane >> 4 & 1) << 1);
      const int u = token(t0);
      transfer(x + (int64_t)u * stride + (uint32_t)((min(u + row, len - 1) - u) * stride + piece * 8) + col, smem + AT_X + wave * 4096 + k * 1024);
    }
  };
  const uint32_t lds = lds_address(smem);
  const uint32_t steps = lds + AT_S + wave * STEP, xbase = lds + AT_X + wave * 4096, xa = (4 * g + (r16 >> 2)) * 64 + (((r16 & 3) >> 1 ^ (g & 1) << 1) << 4) + (r16 & 1) * 8;
  const uint32_t row_at = r16 * RB + ((g ^ swizzle(r16)) << 4), col_at = (4 * g + (r16 >> 2)) * RB + (((r16 & 3) ^ swizzle(4 * g + (r16 >> 2))) << 4);
  const uint32_t wat = lds + AT_W + of * 12 * 1024 + lane * 16;
  // d as a diagonal: the operand that adds d x (exact) for the even and the odd token tiles of 32 keys
  u32x4 skip[2] = {};
  if constexpr (OUT) {
    const uint32_t d = ((const T *)p.d)[head];
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
      for (int e = 0; e < 2; ++e) skip[o][2 * o + e] = r16 == 4 * g + 2 * e ? d : r16 == 4 * g + 2 * e + 1 ? d << 16 : 0u;
  }

  // what a chunk's transfers and stores count behind its first half of x: the second half of x, the stores, the next chunk's b and c and step sizes
  constexpr int STORES = OUT ? 4 : 0;
  // ---- the state: tile i of rows, column tile pt; tiles 2 s and 2 s + 1 together hold rows 32 s + 8 g .. + 7 in lane group g
  f32x4 st[2 * NK][2];
  constexpr int HSIZE = N * P;

  for (;;) {   // the sequences of the row (STATES: the one that goes on behind it)
  const int first = max(lo, start), q0 = p.cu_q[seq], all = p.cu_q[seq + 1] - q0, from = (first - start) * L;
  len = min((hi - first) * L, all - from);
  const int before = p.cu_k[seq + 1] - p.cu_k[seq] - all, slot = p.state_slots[seq];
  const bool keep = slot >= 0 && slot < p.slots, comes = from == 0 && keep && before > 0;   // (with a state of the pool's)
  // this lane's numbers: of the pool's state of the head; of a row's (offsets made anew for each sequence: kept over all of them they are 60 registers)
  int lane_at = g * 8 * P + half * 32 + r16, part_lane = (half * 128 + lane) * 4;
  asm volatile("" : "+v"(lane_at), "+v"(part_lane));
  auto pool = [&](int which) { return p.ssm_state + ((int64_t)which * p.slots + (keep ? slot : 0)) * size + (int64_t)head * HSIZE; };
  auto state_at = [&](int i, int pt, int e) { return lane_at + (i >> 1) * 32 * P + ((i & 1) * 4 + e) * P + pt * 16; };
  auto part = [&](float *of_rows, int row, int i, int pt) { return (f32x4 *)(of_rows + ((int64_t)row * p.heads + head) * HSIZE + part_lane + i * 1024 + pt * 256); };
  x = (const T *)p.x + (int64_t)(q0 + from) * p.x_stride;
  fetch_bc(0);
  const float *ahead = sg.steps + ((int64_t)first * p.heads + head) * 2 * L + lane;   // of the next chunk
  float next_r = ahead[0], next_step = ahead[L];
  fetch_x(0, 0);
  fetch_x(0, 1);
#pragma unroll
  for (int i = 0; i < 2 * NK; ++i)
#pragma unroll
    for (int pt = 0; pt < 2; ++pt) {
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
      if (comes) {
        // (the pool's state of a sequence that goes on in the next row is read by the first launch alone: the second may write it)
        if (OUT && end > hi) {
          v = *part(sg.first, blockIdx.y, i, pt);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = pool(before & 1)[state_at(i, pt, e)];
        }
        if (!OUT) *part(sg.first, blockIdx.y, i, pt) = v;
      }
      st[i][pt] = v;
    }
  if constexpr (OUT) {
    if (from > 0)
      for (int z = start / run; z < (int)blockIdx.y; ++z) {
        const float decay = __builtin_amdgcn_exp2f(sg.decays[(int64_t)z * p.heads + head]);
#pragma unroll
        for (int i = 0; i < 2 * NK; ++i)
#pragma unroll
          for (int pt = 0; pt < 2; ++pt) {
            const f32x4 v = *part(sg.states, z, i, pt);
#pragma unroll
            for (int e = 0; e < 4; ++e) st[i][pt][e] = fmaf(st[i][pt][e], decay, v[e]);
          }
      }
  }

  vm_wait<0>();
  for (int t0 = 0; t0 < len; t0 += L) {
    float tail, over1 = 0.f, over2 = 0.f;   // decays of the chunk, of the second and of the third token tile
    {   // ---- step sizes and decays, a lane a token
      const float r = next_r, step = next_step;
      const float r4 = u2f(__builtin_amdgcn_readlane(f2u(r), 63));
      tail = __builtin_amdgcn_exp2f(r4);
      lds_write32<S_W>(steps + lane * 4, __builtin_amdgcn_exp2f(r4 - r) * step);
      if constexpr (OUT) {
        const float r1 = u2f(__builtin_amdgcn_readlane(f2u(r), 15)), r2 = u2f(__builtin_amdgcn_readlane(f2u(r), 31));
        const float r3 = u2f(__builtin_amdgcn_readlane(f2u(r), 47));
        const float ahead = g == 0 ? 0.f : g == 1 ? r1 : g == 2 ? r2 : r3, last = g == 0 ? r1 : g == 1 ? r2 : g == 2 ? r3 : r4;
        over1 = __builtin_amdgcn_exp2f(r2 - r1), over2 = __builtin_amdgcn_exp2f(r3 - r2);
        lds_write32<S_R>(steps + lane * 4, r);
        lds_write32<S_DT>(steps + lane * 4, step);
        lds_write32<S_ALL>(steps + lane * 4, __builtin_amdgcn_exp2f(r));
        lds_write32<S_E>(steps + lane * 4, __builtin_amdgcn_exp2f(r - ahead));
        lds_write32<S_G>(steps + lane * 4, __builtin_amdgcn_exp2f(last - r) * step);
      } else {
        decayed += r4;
      }
    }
    // this chunk's b and c have landed (behind them: x, stores); every wave is done with the chunk before
    vm_wait<4 + STORES>();
    lds_barrier();
    fetch_bc(t0 + L);   // (behind the end: rows that nobody reads)
    if (t0 + L < len) ahead += p.heads * 2 * L;   // (behind the end: anything)
    next_r = ahead[0], next_step = ahead[L];
    asm volatile("" ::: "memory");
    const uint32_t bc = lds + (t0 / L & 1) * BC;
    uint32_t rows[NK];
#pragma unroll
    for (int s = 0; s < NK; ++s) rows[s] = bc + (row_at ^ (s << 6));

    f32x4 y[4][2];
    if constexpr (OUT) {
      // ---- weighted scores [key][token] of two of the head's token tiles
      auto score = [&](auto I) __attribute__((always_inline)) {
        constexpr int it = decltype(I)::value;
        u32x4 fr[2][it + 2];
        auto ask = [&](auto S) __attribute__((always_inline)) {
          constexpr int s = decltype(S)::value;
          lds_read128<ROWS + it * 16 * RB>(fr[s & 1][0], rows[s]);
          static_for<it + 1>([&](auto J) { lds_read128<decltype(J)::value * 16 * RB>(fr[s & 1][1 + decltype(J)::value], rows[s]); });
        };
        f32x4 sc[it + 1];
#pragma unroll
        for (int j = 0; j <= it; ++j) sc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        float r_tok, e_tok;
        u32x4 gk[it ? it : 1], rk, dk;
        ask(std::integral_constant<int, 0>{});
        static_for<NK>([&](auto S) {
          constexpr int s = decltype(S)::value, newer = s + 1 < NK ? it + 2 : 4 + it;
          if constexpr (s + 1 < NK) {
            ask(std::integral_constant<int, s + 1>{});
          } else {
            lds_read32<S_R + it * 64>(r_tok, steps + r16 * 4);
            lds_read32<S_E + it * 64>(e_tok, steps + r16 * 4);
            static_for<it>([&](auto J) { lds_read128<S_G + decltype(J)::value * 64>(gk[decltype(J)::value], steps + g * 16); });
            lds_read128<S_R + it * 64>(rk, steps + g * 16);
            lds_read128<S_DT + it * 64>(dk, steps + g * 16);
          }
          static_for<it + 2>([&](auto J) { lds_wait<newer>(fr[s & 1][decltype(J)::value]); });
#pragma unroll
          for (int j = 0; j <= it; ++j) sc[j] = mfma16x16x32<Tag>(fr[s & 1][1 + j], fr[s & 1][0], sc[j]);
        });
        lds_wait<0>(r_tok, e_tok);
        static_for<it>([&](auto J) { lds_wait<0>(gk[decltype(J)::value]); });
        lds_wait<0>(rk, dk);
        // In tiles below the diagonal exp(r_i - r_j) is the product of three decays, each at most 1: from the key to its tile's end, over the tiles between,
        // from the token's tile's start to it
        const f32x4 rks = __builtin_bit_cast(f32x4, rk), dks = __builtin_bit_cast(f32x4, dk);
        float over = e_tok;
        static_for<it>([&](auto J) {
          constexpr int j = it - 1 - decltype(J)::value;
          if constexpr (j + 1 < it) over *= j ? over2 : over1;   // (tile j + 1)
          sc[j] *= __builtin_bit_cast(f32x4, gk[j]) * over;
        });
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float w = __builtin_amdgcn_exp2f(r_tok - rks[e]) * dks[e];
          sc[it][e] = 4 * g + e <= r16 ? sc[it][e] * w : 0.f;
        }
        static_for<it / 2 + 1>([&](auto S) {
          constexpr int s = decltype(S)::value;
          u32x4 hi, lo;
          if constexpr (2 * s + 1 <= it) split44<Tag>(sc[2 * s], sc[2 * s + 1], hi, lo);
          else split44<Tag>(sc[2 * s], f32x4{0.f, 0.f, 0.f, 0.f}, hi, lo);
          lds_write128<operand(it, s) * 1024>(wat, hi);
          lds_write128<(6 + operand(it, s)) * 1024>(wat, lo);
        });
      };
      if (half == 0) {
        score(std::integral_constant<int, 0>{});
        score(std::integral_constant<int, 3>{});
      } else {
        score(std::integral_constant<int, 1>{});
        score(std::integral_constant<int, 2>{});
      }
      // ---- S^T c of all tokens, scaled by exp(r_i); what comes out of LDS is asked for one step ahead
#pragma unroll
      for (int it = 0; it < 4; ++it) y[it][0] = y[it][1] = f32x4{0.f, 0.f, 0.f, 0.f};
      u32x4 c[2][4], hi[2][2], lo[2][2];
      float all_of[4];
      auto ask = [&](auto S) __attribute__((always_inline)) {
        constexpr int s = decltype(S)::value;
        static_for<4>([&](auto I) { lds_read128<ROWS + decltype(I)::value * 16 * RB>(c[s & 1][decltype(I)::value], rows[s]); });
      };
      auto parts = [&](auto S) __attribute__((always_inline)) {
        constexpr int s = decltype(S)::value;
#pragma unroll
        for (int pt = 0; pt < 2; ++pt) split44<Tag>(st[2 * s][pt], st[2 * s + 1][pt], hi[s & 1][pt], lo[s & 1][pt]);
      };
      ask(std::integral_constant<int, 0>{});
      parts(std::integral_constant<int, 0>{});
      static_for<NK>([&](auto S) {
        constexpr int s = decltype(S)::value;
        if constexpr (s + 1 < NK) ask(std::integral_constant<int, s + 1>{});
        else static_for<4>([&](auto I) { lds_read32<S_ALL + decltype(I)::value * 64>(all_of[decltype(I)::value], steps + r16 * 4); });
        static_for<4>([&](auto I) { lds_wait<4>(c[s & 1][decltype(I)::value]); });
        // (the vector unit makes the next parts, or ages the state, while the matrix cores are at these)
        if constexpr (s + 1 < NK) {
          parts(std::integral_constant<int, s + 1>{});
        } else {
#pragma unroll
          for (int i = 0; i < 2 * NK; ++i) st[i][0] *= tail, st[i][1] *= tail;
        }
#pragma unroll
        for (int part = 0; part < 2; ++part)
#pragma unroll
          for (int pt = 0; pt < 2; ++pt)
#pragma unroll
            for (int it = 0; it < 4; ++it) y[it][pt] = mfma16x16x32<Tag>(part ? lo[s & 1][pt] : hi[s & 1][pt], c[s & 1][it], y[it][pt]);
        static_for<16>([&](auto) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x2, s + 1 < NK ? 3 : NK, 0);
        });
      });
      static_for<4>([&](auto I) {
        constexpr int it = decltype(I)::value;
        lds_wait<0>(all_of[it]);
        y[it][0] *= all_of[it], y[it][1] *= all_of[it];
      });
    }
    // ---- sums over 32 keys at a time; the state moves on.  What comes out of LDS is asked for a step ahead
    u32x2 xr[2][2];      // x transposed: [column tile][16 keys]
    u32x4 kw[2], wf[2][4];
    u32x2 bt[2][2][2];   // b transposed: [which][row tile][16 keys]
    auto ask_keys = [&](auto S) __attribute__((always_inline)) {
      constexpr int s = decltype(S)::value;
      // this half of x has landed: behind it are the other half, stores and the next chunk's b, c and steps
      vm_wait<2 + STORES + BCS + 2>();
      static_for<2>([&](auto PT) {
        constexpr int pt = decltype(PT)::value;
        lds_read64_tr<s * 2048>(xr[pt][0], xbase + (xa ^ (pt << 5)));
        lds_read64_tr<s * 2048 + 1024>(xr[pt][1], xbase + (xa ^ (pt << 5)));
      });
      lds_read128<S_W + s * 128>(kw[0], steps + g * 16);
      lds_read128<S_W + s * 128 + 64>(kw[1], steps + g * 16);
    };
    auto ask_b = [&](auto Q) __attribute__((always_inline)) {
      constexpr int q = decltype(Q)::value, s = q / NK;
      static_for<2>([&](auto D) {
        constexpr int d = decltype(D)::value;
        lds_read64_tr<s * 32 * RB + d * 8>(bt[q & 1][d][0], bc + (col_at ^ (q % NK << 6)));
        lds_read64_tr<(s * 32 + 16) * RB + d * 8>(bt[q & 1][d][1], bc + (col_at ^ (q % NK << 6)));
      });
    };
    ask_keys(std::integral_constant<int, 0>{});
    ask_b(std::integral_constant<int, 0>{});
    if constexpr (OUT) {
      lds_barrier();   // the head's scores are there
    } else {
#pragma unroll
      for (int i = 0; i < 2 * NK; ++i) st[i][0] *= tail, st[i][1] *= tail;
    }
    static_for<2>([&](auto S) {
      constexpr int s = decltype(S)::value, WF = OUT ? 2 * (4 - 2 * s) : 0;
      if constexpr (OUT)
        static_for<4>([&](auto I) {
          constexpr int it = decltype(I)::value;
          if constexpr (it >= 2 * s) {
            lds_read128<operand(it, s) * 1024>(wf[0][it], wat);
            lds_read128<(6 + operand(it, s)) * 1024>(wf[1][it], wat);
          }
        });
      static_for<2>([&](auto PT) { lds_wait<WF + 4>(xr[decltype(PT)::value][0], xr[decltype(PT)::value][1]); });
      lds_wait<WF + 4>(kw[0], kw[1]);
      fetch_x(t0 + L, s);
      asm volatile("" ::: "memory");
      u32x4 xf[2], hi[2], lo[2];
#pragma unroll
      for (int pt = 0; pt < 2; ++pt) {
        xf[pt] = join(xr[pt][0], xr[pt][1]);
        float f[8];
        unpack8<Tag>(xf[pt], f);
        split44<Tag>(f32x4{f[0], f[1], f[2], f[3]} * __builtin_bit_cast(f32x4, kw[0]), f32x4{f[4], f[5], f[6], f[7]} * __builtin_bit_cast(f32x4, kw[1]), hi[pt], lo[pt]);
      }
      static_for<NK>([&](auto Q) {
        constexpr int q = s * NK + decltype(Q)::value, newer = decltype(Q)::value + 1 < NK ? 4 : s == 0 ? 10 : 0;
        if constexpr (decltype(Q)::value + 1 == NK && s == 0) ask_keys(std::integral_constant<int, 1>{});
        if constexpr (q + 1 < 2 * NK) ask_b(std::integral_constant<int, q + 1>{});
        static_for<2>([&](auto D) { lds_wait<newer>(bt[q & 1][decltype(D)::value][0], bt[q & 1][decltype(D)::value][1]); });
#pragma unroll
        for (int part = 0; part < 2; ++part)
#pragma unroll
          for (int d = 0; d < 2; ++d)
#pragma unroll
            for (int pt = 0; pt < 2; ++pt) {
              f32x4 &to = st[2 * (q % NK) + d][pt];
              to = mfma16x16x32<Tag>(join(bt[q & 1][d][0], bt[q & 1][d][1]), part ? lo[pt] : hi[pt], to);
            }
      });
      if constexpr (OUT) {
        static_for<4>([&](auto I) {   // (there before the rows of b that were waited for)
          constexpr int it = decltype(I)::value;
          if constexpr (it >= 2 * s) lds_wait<s == 0 ? 10 : 0>(wf[0][it], wf[1][it]);
        });
#pragma unroll
        for (int part = 0; part < 3; ++part)
#pragma unroll
          for (int it = 2 * s; it < 4; ++it)
#pragma unroll
            for (int pt = 0; pt < 2; ++pt) {
              if (part < 2) y[it][pt] = mfma16x16x32<Tag>(xf[pt], wf[part][it], y[it][pt]);
              else if (it / 2 == s) y[it][pt] = mfma16x16x32<Tag>(xf[pt], skip[it & 1], y[it][pt]);
            }
      }
    });
    // ---- out: a lane has columns 4 g .. of both tiles; exchanged, 8 g .. of the 32
    if constexpr (OUT) {
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const int t = t0 + it * 16 + r16;
        u32x2 a = pack_quad<Tag>(y[it][0]), b = pack_quad<Tag>(y[it][1]);
        uint32_t a0 = a.x, a1 = a.y, b0 = b.x, b1 = b.y;
        exchange32(a0, b0), exchange32(a1, b1);
        exchange16(a0, b0), exchange16(a1, b1);
        if (t < len) *(u32x4 *)((T *)p.out + (int64_t)(q0 + from + t) * p.out_stride + col + g * 8) = u32x4{a0, a1, b0, b1};
      }
      asm volatile("" ::: "memory");
    }
  }
  vm_wait<0>();
  if constexpr (!OUT) {
#pragma unroll
    for (int i = 0; i < 2 * NK; ++i)
#pragma unroll
      for (int pt = 0; pt < 2; ++pt) *part(sg.states, blockIdx.y, i, pt) = st[i][pt];
    if (half == 0 && lane == 0) sg.decays[(int64_t)blockIdx.y * p.heads + head] = decayed;
    return;
  } else {
    if (keep && from + len >= all) {
      float *ns = pool((before + all) & 1);
#pragma unroll
      for (int i = 0; i < 2 * NK; ++i)
#pragma unroll
        for (int pt = 0; pt < 2; ++pt)
#pragma unroll
          for (int e = 0; e < 4; ++e) ns[state_at(i, pt, e)] = st[i][pt][e];
    }
    if (end >= hi) return;
    go_on();
    lds_barrier();   // every wave is done with the chunk before
  }
  }
}

// Chunks of a row at least: its start is a load of what its sequence's rows before it add
inline int least_run(int max_q) { return std::max(4, (max_q + 8 * L - 1) / (8 * L)); }
// Rows of workgroups, of which one takes a CU to itself; 0: not for these, the kernel of a head a workgroup is as fast.  us, that one and this, 64 heads of 64 x 128,
// sequences of half to all of the longest: 4 of 3900 206 and 136, of 1900 104 and 78, of 1000 58 and 54; 2 of 1900 61 and 56; 16 of 1900 225 and 216; 8 of 1900 123 and
// 122; 1 of 3900 66 and 79; 32 heads: 8 of 3900 186 and 128, 4 of 1900 66 and 57, 8 of 512 32 and 48; of 64 x 64, 64 heads: 4 of 3900 125 and 101, 8 of 1900 95 and 96.
// The lines below run through those: a row's chunks behind what a start and the second launch take, and the other's work, which in whole sequences is less.
inline int pick_rows(int n_seqs, int total_q, int max_q, int heads, int n) {
  if (total_q < max_q || n_seqs <= 0) return 0;   // (no bound of the rows)
  const int64_t chunks = (int64_t)total_q / L + (n_seqs + 1) / 2, most = std::max(1, 256 / (heads / HEADS)), least = least_run(max_q);
  const int64_t rows = std::min(most, (chunks + least - 1) / least), run = std::max(least, (chunks + rows - 1) / rows);
  const double work = (double)chunks * heads / 64, longest = (max_q + L - 1) / L;
  const double here = n > 64 ? 25 + 8.8 * run : 16 + 7.2 * run;
  const double there = mv_ssm_chunk_cuts(n_seqs, total_q, max_q, heads, P, n) ? (n > 64 ? 14 + 0.9 * work : 17 + 0.55 * work)
                                                                                       : std::max(8 + (n > 64 ? 0.6 : 0.43) * work, (n > 64 ? 3.3 : 2.0) * longest);
  return here < 0.97 * there ? (int)rows : 0;
}

template <typename Tag, int NK>
int launch(const MvSsmArgs &a, int rows, int total_q, void *workspace, hipStream_t stream) {
  const int64_t state = (int64_t)rows * a.heads * a.n * a.p;
  float *states = (float *)workspace, *steps = states + 2 * state;
  const int64_t slots = total_q / L + a.n_seqs;
  const Rows r{states, steps + slots * a.heads * 2 * L, states + state, steps, least_run(a.max_q)};
  const dim3 grid(a.heads / HEADS, (unsigned)rows);
  if (int rc = mv_allow_lds<ssm_heads_kernel<Tag, NK, STATES>>()) return rc;
  hipLaunchKernelGGL((ssm_heads_kernel<Tag, NK, STATES>), grid, dim3(512), (lds_bytes<NK, STATES>()), stream, a, r);
  MV_LAUNCH_CHECK();
  if (int rc = mv_allow_lds<ssm_heads_kernel<Tag, NK, OUTPUTS>>()) return rc;
  hipLaunchKernelGGL((ssm_heads_kernel<Tag, NK, OUTPUTS>), grid, dim3(512), (lds_bytes<NK, OUTPUTS>()), stream, a, r);
  MV_LAUNCH_CHECK();
  return MV_OK;
}

}  // namespace

size_t mv_ssm_heads_workspace(int n_seqs, int total_q, int max_q, int heads, int p, int n) {
  if (p != P || (n != 64 && n != 128) || heads % HEADS) return 0;
  const int rows = pick_rows(n_seqs, total_q, max_q, heads, n);
  return rows ? ((size_t)rows * heads * (2 * n * p + 1) + ((size_t)total_q / L + n_seqs) * heads * 2 * L) * sizeof(float) : 0;
}

int mv_ssm_heads_launch(const MvSsmArgs &a, void *workspace, size_t ws_bytes, int total_q, int dtype, hipStream_t stream) {
  if (a.p != P || (a.n != 64 && a.n != 128) || a.heads / a.groups % HEADS || a.x_stride >= 1 << 24) return MV_E_SHAPE;
  const int rows = pick_rows(a.n_seqs, total_q, a.max_q, a.heads, a.n);
  if (!rows || !workspace || ws_bytes < mv_ssm_heads_workspace(a.n_seqs, total_q, a.max_q, a.heads, a.p, a.n)) return MV_E_SHAPE;
  if (dtype == MV_BF16) return a.n == 64 ? launch<bf16_tag, 2>(a, rows, total_q, workspace, stream) : launch<bf16_tag, 4>(a, rows, total_q, workspace, stream);
  return a.n == 64 ? launch<f16_tag, 2>(a, rows, total_q, workspace, stream) : launch<f16_tag, 4>(a, rows, total_q, workspace, stream);
}
