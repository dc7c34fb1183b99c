// K2 (fp32) — packed varlen causal prefill attention on the fp32 matrix cores (v_mfma_f32_32x32x2_f32: exact products, fp32 sums).
//
// Bound by the matrix cores: a flash tile of 32 keys x 32 queries is 64 of these products at head dim 64 (4096 cycles) beside some 1400 of
// vector arithmetic and 16 KiB of LDS reads.  One workgroup = 64 queries of one head, 32 to a wave, and two waves for the same queries that
// take the tiles in turn and meet at the end: blocks of rows differ in length, and short chains of tiles even them out (128 queries a workgroup, four
// waves, each over all tiles: 179 us where two in turn took 151).  S^T = K Q^T puts a query on a lane (and its partner 32 lanes on), so that the row
// maximum is one exchange and P, as it lies in the accumulators, is the operand of O^T += V^T P^T: register r of lane half h holds key
// 8 (r / 4) + 4 h + r % 4, and V is read in that order.  Rows of O^T are dealt so that D / 32 adjacent dims of a key are one read of V and one piece of
// an output row.  The rows of K come into LDS while the products of V run, those of V while the scores do: one set of registers holds them.
//
// Sums are short chains of products, added up like a tree, and a score is scaled where its exponent is formed: as far from 64 bits as the vector kernel
// for rows of a few tokens, nearer for longer ones.  Relative error, this / the vector kernel, 1e-7 (unit normal inputs):
//   head dim 64:  20 tokens 0.81 / 0.81, 50 0.95 / 0.97, 300 1.18 / 1.32, 1000 1.36 / 1.73     (chains of 16 products: 0.92, 1.10, 1.35, 1.50)
//   head dim 128: 20 tokens 0.84 / 0.85, 50 0.99 / 1.05, 300 1.20 / 1.59, 1000 1.37 / 2.26     (chains of 32: 1.05, 1.28, 1.73, 2.25)
// What the tree costs and gives, attention of a layer (us): 6131 tokens in 8 prompts, 12 heads of 64: vector kernel 801, chains of 16 products 137, this
// 148 (62 TFLOP/s of visible pairs; 4 x 2048: 91); 16 x 1024, 16 heads of 128: 958 -> 771 (89), where the longer chains and rows of K and V
// side by side left 69 registers in memory; now 4 (paged or masked: 12; head dim 64: 6).  Whole prompts of head dim 64 have a kernel of their own by now (below).
// The vector kernel (prefill_simple.hip: a wave per query and head, every query reads its keys again) stays for head dim 256, and where queries see few
// keys or are few themselves: vector_is_quicker below.
// Reference: minivllm/models/layers/attention.py:467-504,554-597.
#include "parts.h"
#include "prefill_row.h"

namespace {

constexpr int BN = 32, WAVES = 4, GROUPS = 2, TURNS = WAVES / GROUPS, BM = GROUPS * 32;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) int i32x4;

// first key of its own that a position sees (chunk or window)
__device__ __forceinline__ int first_key_of(const PrefillParams &p, int pos) {
  return p.chunk > 0 ? max(pos, 0) / p.chunk * p.chunk : p.mask.window > 0 ? max(0, pos - p.mask.window + 1) : 0;
}

// GENERAL: paged keys, a window, chunks, capped scores; else whole prompts, keys side by side
template <int D, bool GENERAL>
__global__ void __launch_bounds__(WAVES * 64, D == 64 ? 3 : 2) prefill_f32_kernel(PrefillParams p) {
  constexpr int CPR = D / 4, PER = TURNS * BN * CPR / (WAVES * 64), DT = D / 32;   // 16-byte pieces of a row, of a thread; tiles of 32 dims
  // head dim 64 has the registers to add a chain of products up while the next one runs, and to add two chains of keys to each other first
  constexpr bool BEHIND = D == 64, PAIRS = D == 64;
  constexpr bool QL = D == 64;   // queries in LDS (at head dim 128 they would halve the workgroups of a CU)
  typedef __attribute__((ext_vector_type(DT))) float fdt;
  __shared__ __attribute__((aligned(16))) f32x4 tiles_lds[2][TURNS * BN * CPR];   // K | V
  __shared__ __attribute__((aligned(16))) int there[TURNS][BN];   // (paged) a key has a page
  __shared__ __attribute__((aligned(16))) f32x4 qs[QL ? BM * CPR : 1];
  __shared__ int wild[WAVES];                                     // a wave has put values of V that are not finite
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, col = lane & 31, half = lane >> 5;
  const int group = wave % GROUPS, turn = wave / GROUPS;
  f32x4 *ks = tiles_lds[0], *vs = tiles_lds[1];
  const int head = blockIdx.x, seq = blockIdx.y, hkv = head / (p.n_heads / p.n_kv_heads);
  const int q0 = p.cu_q[seq], sq = p.cu_q[seq + 1] - q0, k0 = p.cu_k[seq], sk = p.cu_k[seq + 1] - k0;
  const int qb = ((int)gridDim.z - 1 - (int)blockIdx.z) * BM;   // the longest rows first
  if (qb >= sq) return;
  const int keep = GENERAL ? p.mask.keep_first : 0;
  const bool paged = GENERAL && p.block_tables != nullptr;
  auto first_key = [&](int at) __attribute__((always_inline)) { return GENERAL ? first_key_of(p, at) : 0; };
  // positions of the workgroup's, the wave's and the lane's queries (queries behind the end repeat the last one)
  const int shift = sk - sq, last = min(qb + BM, sq) - 1;
  const int wq = min(qb + group * 32, sq - 1), qi = min(qb + group * 32 + col, sq - 1), pos = qi + shift;
  const int wave_lo = wq + shift, wave_hi = min(qb + group * 32 + 31, sq - 1) + shift;
  const int first = first_key(pos);
  // tiles [0, heads) hold the kept first keys, tiles [from, to) the rest
  const int end = min(sk, last + shift + 1), to = end > 0 ? (end + BN - 1) / BN : 0;
  const int from = min(first_key(qb + shift) / BN, to), heads = min((min(keep, sk) + BN - 1) / BN, from);
  const int tiles = heads + to - from;
  auto tile_at = [&](int i) __attribute__((always_inline)) { return i < heads ? i : from + i - heads; };

  const float *qp = (const float *)p.q + (int64_t)(q0 + qi) * p.q_stride + (int64_t)head * D + half * (D / 2);
  f32x4 q[QL ? 1 : CPR / 2];   // dims half * D / 2 .. of the lane's query
  f32x4 *qt = qs + group * BM / GROUPS * CPR + col * CPR;
#pragma unroll
  for (int j = 0; j < CPR / 2; ++j) {
    const f32x4 w = *(const f32x4 *)(qp + 4 * j);
    if constexpr (QL) qt[(half * (CPR / 2) + j) ^ (col & 15)] = w;   // (the two waves of a group write the same; a wave reads what it wrote)
    else q[j] = w;
  }

  f32x4 raw[PER];   // rows on their way to LDS: K during the products of V, V during the scores
  unsigned pages = 0;   // bit n: piece n has one
  // (addresses are worked out at each tile: kept, they take the registers of a chain of products)
  auto anew = [](unsigned x) __attribute__((always_inline)) {
    asm volatile("" : "+v"(x));
    return x;
  };
  constexpr int STEP = WAVES * 64 / CPR;   // rows from one piece of a thread to its next
  auto fetch = [&](int i0, const void *rows, const void *cache, int64_t stride) __attribute__((always_inline)) {
    const unsigned here = anew(tid);
    const int row = here / CPR, c = here % CPR;
#pragma unroll
    for (int n = 0; n < PER; ++n) {
      const int from = tile_at(min(i0 + n * STEP / BN, tiles - 1)) * BN;
      const int in = min(row + n * STEP % BN, sk - 1 - from);   // (clamped rows are masked)
      if (!paged) {
        raw[n] = *(const f32x4 *)((const float *)rows + (int64_t)(k0 + from) * stride + (int64_t)hkv * D + (in * stride + 4 * c));
      } else {
        const int key = from + in, bi = key / p.block_size, blk = bi < p.table_width ? p.block_tables[(int64_t)seq * p.table_stride + bi] : -1;
        const bool is = blk >= 0 && blk < p.num_blocks;
        const int64_t at = (is ? (int64_t)blk * p.block_size : 0) + (key - bi * p.block_size);
        pages = n == 0 ? is : pages | (unsigned)is << n;
        raw[n] = *(const f32x4 *)((const float *)cache + (at * p.n_kv_heads + hkv) * D + 4 * c);
      }
    }
    if (paged) {
#pragma unroll
      for (int n = 0; n < PER; ++n)
        if (!(pages >> n & 1)) raw[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  auto fetch_k = [&](int i0) __attribute__((always_inline)) { fetch(i0, p.k, p.k_cache, p.k_stride); };
  auto fetch_v = [&](int i0) __attribute__((always_inline)) { fetch(i0, p.v, p.v_cache, p.v_stride); };
  auto put_k = [&]() __attribute__((always_inline)) {   // in an order that spreads the rows over the banks
    const unsigned here = anew(tid);
    const int row = here / CPR, c = here % CPR;
#pragma unroll
    for (int n = 0; n < PER; ++n) {
      ks[(row + n * STEP) * CPR + (c ^ ((row + n * STEP) & 15))] = raw[n];
      if (paged && c == 0) there[n * STEP / BN][row + n * STEP % BN] = pages >> n & 1;
    }
  };
  auto put_v = [&]() __attribute__((always_inline)) {
    float z = 0.f;
#pragma unroll
    for (int n = 0; n < PER; ++n) {
      vs[tid + n * WAVES * 64] = raw[n];
#pragma unroll
      for (int e = 0; e < 4; ++e) z = fmaf(raw[n][e], 0.f, z);
    }
    const int any = __any(z != 0.f) ? 1 : 0;   // (NaN)
    if (lane == 0) wild[wave] = any;
  };

  const float scale_log2 = p.scale * 1.4426950408889634f;
  const float cap = GENERAL ? p.mask.softcap : 0.f, to_cap = cap > 0.f ? p.scale / cap : 0.f, cap_log2 = cap * 1.4426950408889634f;
  // scores are multiplied by `mul` where their exponent is formed, without a rounding between
  const bool late = !(cap > 0.f) && scale_log2 > 0.f;
  const float mul = late ? scale_log2 : 1.f;
  float m = -1e30f, l = 0.f;
  int apart = 0;   // a tile with masked keys holds values of V that are not finite
  if (p.mask.sink) sink_start(((const float *)p.mask.sink)[head], half == 0 && turn == 0, m, l);
  f32x16 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[t][r] = 0.f;

  if (tiles > 0) {
    fetch_k(0);
    put_k();
    fetch_v(0);
  }
  for (int i0 = 0; i0 < tiles; i0 += TURNS) {
    __syncthreads();   // K is there; every wave is done with V of the tiles before
    put_v();
    const bool more = i0 + TURNS < tiles;
    if (more) fetch_k(i0 + TURNS);
    const int tile = tile_at(min(i0 + turn, tiles - 1)), key0 = tile * BN;
    const f32x4 *kt = ks + turn * BN * CPR, *vt = vs + turn * BN * CPR;
    // of the wave's queries sees a key of it
    const bool some = i0 + turn < tiles && key0 <= wave_hi && (key0 + BN > first_key(wave_lo) || key0 < keep);
    bool masked = false;
    f32x16 s;
    if (some) {
      // A score's D products in chains of eight, four chains to a group, (0 + 1) + (2 + 3)
      const int swizzle = anew(col & 15);
      f32x16 group, pair, before;
      auto join = [&](int c, const f32x16 &x) __attribute__((always_inline)) {
        if (c % 4 == 0) group = x;
        else if (c % 4 == 1) group += x;
        else if (c % 4 == 2) pair = x;
        else group += pair + x;
        if (c % 4 == 3) s = c == 3 ? group : s + group;
        // (here, not where the sum is used: a chain's registers are free)
        if (c % 4 == 2) asm volatile("" : "+v"(pair));
        else asm volatile("" : "+v"(group));
        if (c % 4 == 3) asm volatile("" : "+v"(s));
      };
#pragma unroll
      for (int c = 0; c < CPR / 2; ++c) {
        const int at = (half * (CPR / 2) + c) ^ swizzle;
        const f32x4 k = kt[col * CPR + at], w = QL ? qt[at] : q[QL ? 0 : c];
        f32x16 chain = {};
#pragma unroll
        for (int e = 0; e < 4; ++e) chain = __builtin_amdgcn_mfma_f32_32x32x2f32(k[e], w[e], chain, 0, 0, 0);
        if (!BEHIND) join(c, chain);
        else if (c > 0) join(c - 1, before);
        before = chain;
      }
      if (BEHIND) join(CPR / 2 - 1, before);
      if (cap > 0.f) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = capped_log2<f32_tag>(s[r], to_cap, cap_log2);
      } else if (!late) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] *= scale_log2;
      }
      masked = paged || key0 + BN - 1 > wave_lo || key0 + BN > sk || key0 < first_key(wave_hi);
      if (masked) {   // register r of lane half h holds key 8 (r / 4) + 4 h + r % 4 of the tile
        const int upto = min(pos, sk - 1) - key0 - 4 * half, since = first - key0 - 4 * half, kept = keep - key0 - 4 * half;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          i32x4 is = {1, 1, 1, 1};
          if (paged) is = *(const i32x4 *)&there[turn][8 * c + 4 * half];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int j = 8 * c + e;
            s[4 * c + e] = j <= upto && (!GENERAL || j >= since || j < kept) && is[e] ? s[4 * c + e] : -INFINITY;
          }
        }
      }
    }
    __syncthreads();   // V is there; every wave is done with K
    if (more) {
      put_k();
      fetch_v(i0 + TURNS);
    }
    if (some) {
      if (masked) apart |= wild[0] | wild[1] | wild[2] | wild[3];
      float mx = s[0];
#pragma unroll
      for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
      mx = fmaxf(m, fmaxf(mx, __shfl_xor(mx, 32, 64)) * mul);
      if (__any(mx > m)) {
        const float alpha = __builtin_amdgcn_exp2f(m - mx);
        l *= alpha;
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[t][r] *= alpha;
        m = mx;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], mul, -m));
      l += (((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]))) + (((s[8] + s[9]) + (s[10] + s[11])) + ((s[12] + s[13]) + (s[14] + s[15])));
      // the keys apart from the sums so far, in chains of eight; of four where rows may have few
      auto values = [&](auto N) __attribute__((always_inline)) {
        constexpr int M = decltype(N)::value;
        f32x16 before, part[DT];
        auto join = [&](int i, const f32x16 &x) __attribute__((always_inline)) {
          const int c = i / DT, t = i % DT;
          if (PAIRS && M == 2 && c % 2 == 0) {
            part[t] = x;
            return;
          }
          o[t] += PAIRS && M == 2 ? part[t] + x : x;
          asm volatile("" : "+v"(o[t]));
        };
#pragma unroll
        for (int c = 0; c < 16 / M; ++c) {
          fdt v[M];
#pragma unroll
          for (int r = 0; r < M; ++r) v[r] = ((const fdt *)vt)[(8 * ((c * M + r) >> 2) + 4 * half + ((c * M + r) & 3)) * 32 + col];
#pragma unroll
          for (int t = 0; t < DT; ++t) {
            f32x16 sums = {};
#pragma unroll
            for (int r = 0; r < M; ++r) sums = __builtin_amdgcn_mfma_f32_32x32x2f32(v[r][t], s[M * c + r], sums, 0, 0, 0);
            if (!BEHIND) join(c * DT + t, sums);
            else if (c + t > 0) join(c * DT + t - 1, before);
            before = sums;
          }
        }
        if (BEHIND) join(16 / M * DT - 1, before);
      };
      if (masked) values(std::integral_constant<int, 2>{});
      else values(std::integral_constant<int, 4>{});
    }
  }
  // the second wave of each query group hands its part over
  __syncthreads();
  float *part = (float *)tiles_lds + group * 64 * (16 * DT + 2) + lane;
  if (lane == 0) wild[wave] = apart;
  if (turn > 0) {
    part[0] = m, part[64] = l;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) part[64 * (2 + 16 * t + r)] = o[t][r];
  }
  __syncthreads();
  if (turn > 0) return;
  if (wild[group] | wild[group + GROUPS]) {   // 0 x infinity of a masked key is in the sums: these rows again, key by key
    for (int t = qb + group * 32; t < min(qb + group * 32 + 32, sq); ++t) prefill_row<f32_tag, D>(p, seq, q0 + t, head);
    return;
  }
  {
    const float m1 = part[0], mx = fmaxf(m, m1), f0 = __builtin_amdgcn_exp2f(m - mx), f1 = __builtin_amdgcn_exp2f(m1 - mx);
    l = l * f0 + part[64] * f1;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[t][r] = o[t][r] * f0 + part[64 * (2 + 16 * t + r)] * f1;
  }
  l += __shfl_xor(l, 32, 64);
  // a lane's rows 8 a + 4 half + b of tile t are dims DT (8 a + 4 half + b) + t: 4 DT adjacent ones for each a
  const bool mine = qb + group * 32 + col < sq;
  const int64_t token = q0 + qi;
  float *op = (float *)p.out + token * p.out_stride + (int64_t)head * D;
  if (mine) {
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int c = 0; c < DT; ++c) {
        const int dim = DT * (8 * a + 4 * half) + 4 * c;
        f32x4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = o[(4 * c + e) % DT][4 * a + (4 * c + e) / DT];
          w[e] = l > 0.f ? x / l * attn_factor<f32_tag>(p.mask, token, head * D + dim + e) : 0.f;
        }
        *(f32x4 *)(op + dim) = w;
      }
  }
}

// ---- whole prompts, keys side by side, head dim 64: the same tiles by parts of bf16 (parts.h), a product the six of its parts' products that matter.
// 32 queries to a wave, K and V brought into parts on their way into LDS, for 128 queries at a time, or for 64, whose waves take 32 keys each of 64 in turn and meet
// at the end, where there are not enough of the larger ones.  S^T = K Q^T puts four keys of a query in a lane, and P, as it lies in the accumulators, is the
// operand of O^T += V^T P^T, whose V is read transposed in that order of keys.  Of a score's products and of a tile of values the smallest are added up first, and 32 keys'
// values apart from the rest, so that one sum in 32 keys rounds at its size.  What is not finite goes to the vector kernel's rows.
// Bound by vector arithmetic and products that do not overlap enough (58 + 40 % of the CUs' cycles): 200 instructions for the softmax and P's parts of 32 x 32, 120 for those
// of K and V, beside 96 products.  us, the fp32 products' kernel / 64 queries / 128: 12 heads, 8 prompts of 511 .. 1021 tokens 141 / 90 / 83 (and the distance
// from 64 bits 1.31e-7, 1.08, 1.10); one of 1000 64 / 44 / 63; 4 of 2048 283 / 177 / 159; 80 of 50 26 / 22 / 25.  Tried: v_dot2_f32_bf16 for the rests 86 (128 queries), two tiles of values
// at a time 82, values' products straight into the sums 82 and 2.0e-7, priority for the products 82.
typedef __attribute__((ext_vector_type(2))) uint16_t u16x2;
// the largest bits of first parts, those of numbers that are too large and of what is not finite among them
constexpr uint32_t kTooLarge = (127 + 104) << 7;
__device__ __forceinline__ void look(const u32x4 &first, u16x2 &odd) {
#pragma unroll
  for (int i = 0; i < 4; ++i) odd = __builtin_elementwise_max(odd, __builtin_bit_cast(u16x2, first[i] & 0x7fff7fffu));
}
__device__ __forceinline__ u32x2 read_tr(const char *p) {
  typedef __attribute__((ext_vector_type(4))) short s16x4;
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)p));
}
// Below 2^-109 three of bf16 do not add up to a number of fp32.  Values and probabilities are taken times 2^16, so that none is without its last bits.  What queries and
// keys lose, 2^-134 at the most, is 2^-24 of a score's unit beside the largest that are taken (2^104; values: 2^88), and larger ones go the other way.
// Costs 2 %: 8 prompts of 511 .. 1021 tokens 81.1 -> 83.0 us, 4 of 2048 164 -> 169.
constexpr float kValues = 0x1p16f;
__device__ __forceinline__ f32x4 mfma(const u32x4 &a, const u32x4 &b, const f32x4 &c) { return mfma16x16x32<bf16_tag>(a, b, c); }

template <int D, int GROUPS>   // (head dim 128: 55 registers in memory; 8 prompts of 511 .. 1021 tokens 255 -> 201 us, one of 1000 111 -> 157)
__global__ void __launch_bounds__(256, 2) prefill_parts_kernel(PrefillParams p) {
  constexpr int TURNS = 4 / GROUPS, BM = 32 * GROUPS, BN = 4096 / D, SUBS = BN / 32 / TURNS, KS = D / 32, DT = D / 16, CH = D / 8;   // (32 keys: a sub)
  constexpr int PART = BN * D * 2;
  static_assert(SUBS >= 1 && D == 64);
  __shared__ __attribute__((aligned(16))) char kl[3 * PART], vl[3 * PART];
  __shared__ int again;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r16 = lane & 15, g = lane >> 4, group = wave % GROUPS, turn = wave / GROUPS;
  const int head = blockIdx.x, seq = blockIdx.y, hkv = head / (p.n_heads / p.n_kv_heads);
  const int q0 = p.cu_q[seq], sq = p.cu_q[seq + 1] - q0, k0 = p.cu_k[seq], sk = p.cu_k[seq + 1] - k0;
  const int qb = ((int)gridDim.z - 1 - (int)blockIdx.z) * BM;   // the longest rows first
  if (qb >= sq) return;
  if (tid == 0) again = 0;
  const int shift = sk - sq, last = min(qb + BM, sq) - 1, end = min(sk, last + shift + 1), steps = end > 0 ? (end + BN - 1) / BN : 0;
  const int wave_lo = min(qb + group * 32, sq - 1) + shift, wave_hi = min(qb + group * 32 + 31, sq - 1) + shift;
  // places of a row's pieces of eight, in orders that spread the rows that are read together over the banks
  auto k_place = [](int row, int c) { return (row * CH + (c ^ (row >> 1 & 7))) * 16; };
  auto v_place = [](int row, int c) { return (row * CH + (c ^ (row & 6))) * 16; };

  f32x4 raw[2][2][2];   // rows of K, V on their way
  auto fetch = [&](int step) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const int at = tid + n * 256, row = min(step * BN + at / CH, sk - 1), c = at % CH * 8;   // (rows behind the end: the last one again, masked)
      const float *k = (const float *)p.k + (int64_t)(k0 + row) * p.k_stride + (int64_t)hkv * D + c, *v = (const float *)p.v + (int64_t)(k0 + row) * p.v_stride + (int64_t)hkv * D + c;
      raw[0][n][0] = *(const f32x4 *)k, raw[0][n][1] = *(const f32x4 *)(k + 4);
      raw[1][n][0] = *(const f32x4 *)v, raw[1][n][1] = *(const f32x4 *)(v + 4);
    }
  };
  u16x2 odd = {0, 0};
  auto put = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const int at = tid + n * 256, row = at / CH, c = at % CH;
        const f32x4 &a = raw[w][n][0], &b = raw[w][n][1];
        const float by = w ? kValues : 1.f;
        float f[8] = {a[0] * by, a[1] * by, a[2] * by, a[3] * by, b[0] * by, b[1] * by, b[2] * by, b[3] * by};
        u32x4 part[3];
        split3<false>(f, part);
        look(part[0], odd);
#pragma unroll
        for (int s = 0; s < 3; ++s) *(u32x4 *)((w ? vl : kl) + s * PART + (w ? v_place(row, c) : k_place(row, c))) = part[s];
      }
  };
  if (steps > 0) fetch(0);
  u32x4 q[2][KS][3];   // dims 32 s + 8 g .. of query 16 i + r16
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const float *from = (const float *)p.q + (int64_t)(q0 + min(qb + group * 32 + i * 16 + r16, sq - 1)) * p.q_stride + (int64_t)head * D + s * 32 + g * 8;
      const f32x4 a = *(const f32x4 *)from, b = *(const f32x4 *)(from + 4);
      float f[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
      split3<false>(f, q[i][s]);
      look(q[i][s][0], odd);
    }
  const float scale_log2 = p.scale * 1.4426950408889634f;
  const bool late = scale_log2 > 0.f;   // scores are multiplied by `mul` where their exponent is formed, without a rounding between
  const float mul = late ? scale_log2 : 1.f;
  float m[2] = {-1e30f, -1e30f}, l[2] = {0.f, 0.f};
  if (p.mask.sink)
#pragma unroll
    for (int i = 0; i < 2; ++i) sink_start(((const float *)p.mask.sink)[head], g == 0 && turn == 0, m[i], l[i]);
  f32x4 o[2][DT] = {};   // dims 16 t + 4 g .. of query 16 i + r16
  for (int step = 0; step < steps; ++step) {
    __syncthreads();   // every wave is done with the keys before
    put();
    if (step + 1 < steps) fetch(step + 1);
    __syncthreads();
#pragma unroll
    for (int sub = 0; sub < SUBS; ++sub) {
      const int in = (TURNS == 1 ? sub : turn) * 32, key0 = step * BN + in;
      if (key0 > wave_hi || key0 >= sk) continue;   // (of the wave)
      // scores, keys by queries: the smallest products first, so that only the last of a row's KS sums round at its size
      f32x4 s[2][2] = {};
      const char *kt = kl;
#pragma unroll
      for (int c = 0; c < KS; ++c) {
        u32x4 k[2][3];
#pragma unroll
        for (int b = 0; b < 3; ++b)
#pragma unroll
          for (int j = 0; j < 2; ++j) k[j][b] = *(const u32x4 *)(kt + b * PART + k_place(in + 16 * j + r16, 4 * c + g));
#pragma unroll
        for (int b = 2; b >= 1; --b)
#pragma unroll
          for (int a = 0; a <= b; ++a)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
              for (int i = 0; i < 2; ++i) s[j][i] = mfma(k[j][a], q[i][c][b - a], s[j][i]);
      }
#pragma unroll
      for (int c = 0; c < KS; ++c) {
        u32x4 k[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) k[j] = *(const u32x4 *)(kt + k_place(in + 16 * j + r16, 4 * c + g));
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int i = 0; i < 2; ++i) s[j][i] = mfma(k[j], q[i][c][0], s[j][i]);
      }
      if (!late)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int i = 0; i < 2; ++i) s[j][i] *= scale_log2;
      if (key0 + 31 > wave_lo || key0 + 32 > sk) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int upto = min(min(qb + group * 32 + i * 16 + r16, sq - 1) + shift, sk - 1) - key0 - 4 * g;
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) s[j][i][e] = 16 * j + e <= upto ? s[j][i][e] : -INFINITY;
        }
      }
      u32x4 w[2][3];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        float mx = fmaxf(fmaxf(fmaxf(s[0][i][0], s[0][i][1]), fmaxf(s[0][i][2], s[0][i][3])), fmaxf(fmaxf(s[1][i][0], s[1][i][1]), fmaxf(s[1][i][2], s[1][i][3])));
        float a, b;
        swap16(mx, a, b);
        swap32(fmaxf(a, b), a, b);
        mx = fmaxf(m[i], fmaxf(a, b) * mul);
        if (__any(mx > m[i])) {
          const float alpha = __builtin_amdgcn_exp2f(m[i] - mx);
          l[i] *= alpha;
#pragma unroll
          for (int t = 0; t < DT; ++t) o[i][t] *= alpha;
          m[i] = mx;
        }
        float f[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = __builtin_amdgcn_exp2f(fmaf(s[e >> 2][i][e & 3], mul, -m[i]));
        l[i] += ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] *= kValues;
        split3<false>(f, w[i]);
      }
      // values: a tile's products of these keys apart, the smallest first, one sum into the rest's
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        u32x4 v[3];
#pragma unroll
        for (int b = 0; b < 3; ++b) {
          const int row = in + 4 * g + (r16 >> 2), c = 2 * t + ((r16 & 3) >> 1);
          const u32x2 lo = read_tr(vl + b * PART + v_place(row, c) + (r16 & 1) * 8), hi = read_tr(vl + b * PART + v_place(row + 16, c) + (r16 & 1) * 8);
          v[b] = u32x4{lo[0], lo[1], hi[0], hi[1]};
        }
        f32x4 sum[2] = {};
#pragma unroll
        for (int b = 2; b >= 0; --b)
#pragma unroll
          for (int a = 0; a <= b; ++a)
#pragma unroll
            for (int i = 0; i < 2; ++i) sum[i] = mfma(v[a], w[i][b - a], sum[i]);
#pragma unroll
        for (int i = 0; i < 2; ++i) o[i][t] += sum[i];
      }
    }
  }
  // what the turns have of the same queries together; numbers that are not finite anywhere: these rows again, key by key
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    float a, b;
    swap16(l[i], a, b);
    swap32(a + b, a, b);
    l[i] = a + b;
  }
  bool bad = odd[0] >= kTooLarge || odd[1] >= kTooLarge;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    bad |= !(l[i] < INFINITY);
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) bad |= !(fabsf(o[i][t][e]) < INFINITY);
  }
  __syncthreads();
  if (__any(bad) && lane == 0) again = 1;
  if constexpr (TURNS > 1) {
    float *part = (float *)kl + group * 64 * (2 * DT * 4 + 4) + lane;
    static_assert(GROUPS * 64 * (8 * DT + 4) * 4 <= 3 * PART);
    if (turn > 0) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        part[64 * i] = m[i], part[64 * (2 + i)] = l[i];
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) part[64 * (4 + (i * DT + t) * 4 + e)] = o[i][t][e];
      }
    }
    __syncthreads();
    if (turn == 0) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float m1 = part[64 * i], mx = fmaxf(m[i], m1), f0 = __builtin_amdgcn_exp2f(m[i] - mx), f1 = __builtin_amdgcn_exp2f(m1 - mx);
        l[i] = l[i] * f0 + part[64 * (2 + i)] * f1;
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) o[i][t][e] = o[i][t][e] * f0 + part[64 * (4 + (i * DT + t) * 4 + e)] * f1;
      }
    }
  } else {
    __syncthreads();
  }
  if (again) {
    for (int t = qb + wave; t <= last; t += 4) prefill_row<f32_tag, D>(p, seq, q0 + t, head);
    return;
  }
  if (turn > 0) return;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int at = qb + group * 32 + i * 16 + r16;
    if (at >= sq) continue;
    const int64_t token = q0 + at;
    float *op = (float *)p.out + token * p.out_stride + (int64_t)head * D + 4 * g;
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      f32x4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = l[i] > 0.f ? o[i][t][e] / l[i] * (1.f / (kValues * kValues)) * attn_factor<f32_tag>(p.mask, token, head * D + 16 * t + 4 * g + e) : 0.f;
      *(f32x4 *)(op + 16 * t) = w;
    }
  }
}

// Both kernels' times in ns.  The vector kernel takes 3 us, the walk to the sequence, and 0.11 us a key (twice that at head dim 128) or its reads of K and V,
// whichever is more.
// fp32 products (head dim 128, pages, masks), as they grew over 1700 shapes (1 .. 400 queries of 1 .. 2000 keys, 4 .. 32 heads, 1 .. 256 sequences): a tile of 64
// queries 9 us for the first 64 keys and 4 for each further 64, or what its turns on the chip take.  The other kernel is quicker by more than 5 % in 5 % of them, by 45 % at most.
// Vector kernel / this, us: one prompt of 8 tokens, 12 heads of 128 4 / 15; 64 of 8 tokens 16 / 31, of 16 28 / 32; one of 64 tokens 17 / 15;
// 256 single queries of 400 paged keys, 32 heads of 64 (128) 193 / 953 (349 / 2270).
// Parts (whole prompts of head dim 64), over 3340 shapes (1 .. 1000 tokens, 4 .. 32 heads, 1 .. 128 prompts): 8.5 us for the first 64 keys and 1.7 for each further 64, or its turns.
// The other one is quicker by more than 5 % in 1 %, by 33 % at most (with the fp32 products' figures 5 %, 53 %).  Vector kernel / this, us, 12 heads: one prompt of 8 tokens
// 4.2 / 7.6, 48 8.4 / 8.6, 65 10.5 / 9.6, 87 12.7 / 10.7; 8 of 32 tokens 8.2 / 8.5, of 40 9.8 / 8.7; 64 of 8 tokens, 32 heads 27 / 28.
// From 320 keys on, where the vector kernel is further from 64 bits, it has to take half as long or less.
bool general(const PrefillParams &p) { return p.block_tables || p.chunk > 0 || p.mask.window > 0 || p.mask.softcap > 0.f; }
bool vector_is_quicker(const PrefillParams &p) {
  const int64_t seen = p.max_seqlen_k, wide = p.head_dim / 64, beside = min(p.max_seqlen_q, BM) + BN - 2;   // keys that only other queries of a tile see
  const int64_t limit = p.chunk > 0 ? p.chunk : p.mask.window > 0 ? (int64_t)p.mask.window + p.mask.keep_first : seen;
  const int64_t keys = min(seen, limit), pieces = (min(seen, limit < seen ? limit + beside : seen) + 63) / 64;
  const int64_t rows = (int64_t)p.n_heads * p.n_seqs * p.max_seqlen_q, groups = (int64_t)p.n_heads * p.n_seqs * ((p.max_seqlen_q + BM - 1) / BM);
  const int64_t read = rows * keys * wide / 25 / (p.n_heads >= 4 * p.n_kv_heads ? 2 : 1);
  const int64_t vector = 3000 + 70 * p.n_seqs + max(22 * wide * keys * (p.block_tables ? 6 : 5), read) + rows * p.n_seqs * 14 / 1000;
  const int64_t tiles = wide == 1 && !general(p) ? max(6800 + 1700 * pieces, groups * (10 + 7 * pieces))
                                                 : max(4700 + 4000 * pieces, groups * (7 + 12 * pieces)) * (wide > 1 ? 7 : 4) / 4 *
                                                       (p.block_tables ? 14 : limit < seen || p.mask.softcap > 0.f ? 12 : 10) / 10;
  return vector * (keys > 320 ? 2 : 1) <= tiles;
}

}  // namespace

int mv_prefill_f32_launch(const PrefillParams &p, bool always, hipStream_t stream) {
  if (p.head_dim > 128 || (!always && vector_is_quicker(p))) return MV_E_SHAPE;
  const dim3 grid(p.n_heads, p.n_seqs, (p.max_seqlen_q + BM - 1) / BM);
  if (grid.y > 65535 || grid.z > 65535) return MV_E_SHAPE;
  const dim3 block(WAVES * 64);
  if (p.head_dim == 64 && general(p)) hipLaunchKernelGGL((prefill_f32_kernel<64, true>), grid, block, 0, stream, p);
  else if (p.head_dim == 64) {
    // 128 queries a workgroup where they fill the chip one and a half times (two a CU).  64 / 128 queries, over 130 shapes: 0.67 .. 1.0 of the time up to 600 workgroups of 128,
    // 0.88 .. 1.05 up to 768, 0.91 .. 1.09 up to 1100, 1.0 .. 1.2 over that
    const dim3 wide(p.n_heads, p.n_seqs, (p.max_seqlen_q + 127) / 128);
    if ((int64_t)wide.x * wide.y * wide.z >= 768) hipLaunchKernelGGL((prefill_parts_kernel<64, 4>), wide, block, 0, stream, p);
    else hipLaunchKernelGGL((prefill_parts_kernel<64, 2>), grid, block, 0, stream, p);
  }
  else if (p.head_dim == 128 && general(p)) hipLaunchKernelGGL((prefill_f32_kernel<128, true>), grid, block, 0, stream, p);
  else if (p.head_dim == 128) hipLaunchKernelGGL((prefill_f32_kernel<128, false>), grid, block, 0, stream, p);
  else return MV_E_SHAPE;
  MV_LAUNCH_CHECK();
  return MV_OK;
}
