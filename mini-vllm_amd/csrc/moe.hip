// K17 — mixture of experts (include/mvhip.h): router, grouping of (token, choice) pairs by expert, products over the groups.
//   mv_moe_route:  logits, softmax, choice by groups, weights; 16 or 32 tokens per workgroup;
//   mv_moe_group:  pairs sorted by expert, and the tiles of at most tile_m rows of one expert each;
//   mv_moe_linear: out[place] = W[expert of the place] x[token of the place], with the gate's activation if asked for.
// The weighted sum over a token's choices rides in mv_residual_update.
#include <algorithm>
#include <type_traits>

#include "latent.h"

namespace {

// ---- router ------------------------------------------------------------------------------------------------------------
struct RouteParams {
  const void *x, *w, *correction;
  int32_t *ids;
  float *weights;
  int64_t x_stride;
  int rows, k, outputs, top, groups, keep, flags;
  float scale;
};
constexpr int kRouteTiles = 4;   // tiles of 16 outputs at a time
// grouping by the router's own (only) workgroup
typedef __attribute__((ext_vector_type(4))) int s32x4;
struct RouteGroups {
  int32_t *place, *tokens, *tiles;
  float *by_place;   // or NULL
  int experts, tile_m, max_tiles;
};
constexpr int kRouteRows = 16, kRouteItems = 256, kPairBits = 8;   // (items: pairs and experts, four lanes each)

// largest value of the wave and the lowest index that has it
__device__ __forceinline__ void wave_argmax(float &v, int &i) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float u = __shfl_xor(v, o, 64);
    const int j = __shfl_xor(i, o, 64);
    if (u > v || (u == v && j < i)) v = u, i = j;
  }
}
// lane of the largest value, the lowest one that has it; `free`: lanes that may be chosen (a row of NaN: the first of them)
__device__ __forceinline__ int wave_best(float v, unsigned long long free) {
  const bool mine = free >> (threadIdx.x & 63) & 1;
  const float m = wave_max(mine ? v : -INFINITY);
  const unsigned long long hit = __ballot(mine && v == m);
  return __builtin_ctzll(hit ? hit : free);
}

// the scores of a token's R outputs, in s (logits) and c (scratch): choice and weights, by one wave; `correction`: of output `lane`
template <typename Tag>
__device__ __forceinline__ void choose(const RouteParams &p, float *s, float *c, int64_t token, float correction, int *keys = nullptr, float *weights_too = nullptr) {
  typedef typename elem<Tag>::T T;
  const int lane = threadIdx.x & 63, R = p.outputs, size = R / p.groups;
  const bool sigmoid = p.flags & MV_ROUTE_SIGMOID;
  int mine = 0;
  float weight = 0.f, total = 0.f;
  if (R <= 64 && p.groups <= 8) {   // an output to a lane: nothing goes through LDS
    const bool is = lane < R;
    const float z = is ? s[lane] : -INFINITY;
    float v;
    if (sigmoid) {
      v = 1.0f / (1.0f + expf(-z));
    } else {
      const float mx = wave_max(z), e = is ? expf(z - mx) : 0.f;
      v = e / wave_sum(e);
    }
    const float choice = p.correction ? v + correction : v;
    const unsigned long long all = R == 64 ? ~0ull : (1ull << R) - 1;
    unsigned long long free = all;
    if (p.keep < p.groups) {
      float best = -INFINITY;   // lane = group
      for (int g = 0; g < p.groups; ++g) {
        const float m = wave_max(is && lane / size == g ? choice : -INFINITY);
        if (lane == g) best = m;
      }
      unsigned long long left = (1ull << p.groups) - 1;
      free = 0;
      for (int k = 0; k < p.keep; ++k) {
        const int g = wave_best(best, left);
        left &= ~(1ull << g);
        free |= (size == 64 ? ~0ull : (1ull << size) - 1) << (g * size);
      }
    }
    for (int k = 0; k < p.top; ++k) {
      const int at = wave_best(choice, free);
      free &= ~(1ull << at);
      const float chosen = u2f(__builtin_amdgcn_readlane(f2u(v), __builtin_amdgcn_readfirstlane(at)));
      if (lane == k) mine = at, weight = chosen;
      total += chosen;
    }
  } else {
    float mx = -INFINITY, sum = 0.f;
    if (!sigmoid) {
      for (int i = lane; i < R; i += 64) mx = fmaxf(mx, s[i]);
      mx = wave_max(mx);
      for (int i = lane; i < R; i += 64) sum += expf(s[i] - mx);
      sum = wave_sum(sum);
    }
    for (int i = lane; i < R; i += 64) {
      const float v = sigmoid ? 1.0f / (1.0f + expf(-s[i])) : expf(s[i] - mx) / sum;
      s[i] = v;
      c[i] = p.correction ? v + elem<Tag>::ld(((const T *)p.correction)[i]) : v;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (p.keep < p.groups) {   // lane = group (at most 64)
      float best = -INFINITY;
      if (lane < p.groups)
        for (int i = 0; i < size; ++i) best = fmaxf(best, c[lane * size + i]);
      bool kept = false;
      for (int k = 0; k < p.keep; ++k) {
        float v = kept || lane >= p.groups ? -INFINITY : best;
        int i = kept || lane >= p.groups ? 1 << 20 : lane;
        wave_argmax(v, i);
        if (i == lane) kept = true;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (lane < p.groups && !kept)
        for (int i = 0; i < size; ++i) c[lane * size + i] = -INFINITY;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    for (int k = 0; k < p.top; ++k) {
      float v = -INFINITY;
      int at = 1 << 20;
      for (int i = lane; i < R; i += 64)
        if (c[i] > v || at == 1 << 20) v = c[i], at = i;
      wave_argmax(v, at);
      const float chosen = s[at];
      if (lane == k) mine = at, weight = chosen;
      total += chosen;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (lane == (at & 63)) c[at] = -INFINITY;   // (the lane that looks at it)
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }
  if (lane < p.top) {
    const float w = (p.flags & MV_ROUTE_RAW ? weight : weight / (total + 1e-20f)) * p.scale;
    p.ids[token * p.top + lane] = mine;
    p.weights[token * p.top + lane] = w;
    if (keys) {
      const int pair = (int)token * p.top + lane;
      keys[pair] = mine << kPairBits | pair, weights_too[pair] = w;
    }
  }
}

// The same of four tokens, 16 lanes each, where a wave has that many: output 16 j + l in register j of lane l; at most 64 outputs and 8 groups.  Bits as of
// `choose`: the sums run in its order, a tie goes to the lowest output.  9001 tokens, 34 outputs: this end of a workgroup 6.0 us, four tokens at once 2.3
// (a wave that has one token only: 1.7, at once with three others 2.1).
template <typename Tag>
__device__ __forceinline__ void choose_four(const RouteParams &p, const float *s, int64_t token, bool there, const float (&correction)[4]) {
  const int lane = threadIdx.x & 63, l = lane & 15, R = p.outputs, size = R / p.groups;
  const bool sigmoid = p.flags & MV_ROUTE_SIGMOID;
  bool is[4];
  float v[4], choice[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) is[j] = j * 16 + l < R, v[j] = is[j] ? s[j * 16 + l] : -INFINITY;
  if (sigmoid) {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = 1.0f / (1.0f + expf(-v[j]));
  } else {
    const float mx = row16_max(fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])));
    float sum[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = is[j] ? expf(v[j] - mx) : 0.f, sum[j] = row16_sum(v[j]);
    const float all = (sum[0] + sum[1]) + (sum[2] + sum[3]);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = v[j] / all;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) choice[j] = p.correction ? v[j] + correction[j] : v[j];
  // the lowest index, among those that may be chosen, of the largest value (a row of NaN: the first of them)
  auto best_of = [&](const float *x, auto N, unsigned long long free) {
    constexpr int n = decltype(N)::value;
    float m = -INFINITY, at = -64.f;
#pragma unroll
    for (int j = 0; j < n; ++j) m = fmaxf(m, free >> (j * 16 + l) & 1 ? x[j] : -INFINITY);
    m = row16_max(m);
#pragma unroll
    for (int j = n - 1; j >= 0; --j)
      if ((free >> (j * 16 + l) & 1) && x[j] == m) at = -(float)(j * 16 + l);
    const int i = (int)-row16_max(at);
    return i < 64 ? i : __builtin_ctzll(free);
  };
  unsigned long long free = R == 64 ? ~0ull : (1ull << R) - 1;
  if (p.keep < p.groups) {
    float best = -INFINITY;   // lane = group
    for (int g = 0; g < p.groups; ++g) {
      float m = -INFINITY;
#pragma unroll
      for (int j = 0; j < 4; ++j) m = fmaxf(m, is[j] && j * 16 + l >= g * size && j * 16 + l < (g + 1) * size ? choice[j] : -INFINITY);
      m = row16_max(m);
      if (l == g) best = m;
    }
    unsigned long long left = (1ull << p.groups) - 1;
    free = 0;
    for (int k = 0; k < p.keep; ++k) {
      const int g = best_of(&best, std::integral_constant<int, 1>{}, left);
      left &= ~(1ull << g);
      free |= (size == 64 ? ~0ull : (1ull << size) - 1) << (g * size);
    }
  }
  int mine[4] = {};   // choice 16 j + l
  float weight[4] = {}, total = 0.f;
  for (int k = 0; k < p.top; ++k) {
    const int at = best_of(choice, std::integral_constant<int, 4>{}, free), j = at >> 4;
    free &= ~(1ull << at);
    const float chosen = __shfl(j == 0 ? v[0] : j == 1 ? v[1] : j == 2 ? v[2] : v[3], (lane & 48) + (at & 15), 64);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i * 16 + l == k) mine[i] = at, weight[i] = chosen;
    total += chosen;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (there && i * 16 + l < p.top) {
      p.ids[token * p.top + i * 16 + l] = mine[i];
      p.weights[token * p.top + i * 16 + l] = (p.flags & MV_ROUTE_RAW ? weight[i] : weight[i] / (total + 1e-20f)) * p.scale;
    }
}

// What moe_group_kernel makes of the choices, `pairs` of them in LDS as id << kPairBits | number (a multiple of 16 readable, the largest int behind the last), by one
// workgroup of 16 waves: four lanes to a pair, or behind those to an expert, each counts a quarter of the choices that sort ahead of it.  (One lane each, and choices
// of lower experts, of the same and of those the ones ahead counted apart: 128 pairs took 3 us more than the launch that it saves.)
__device__ __forceinline__ void group_few(const RouteGroups &q, const int *keys, const float *weights, int pairs, int top) {
  const int item = threadIdx.x >> 2, part = threadIdx.x & 3;
  const bool pair = item < pairs;
  const int own = pair ? keys[item] : 0, e = pair ? own >> kPairBits : item - pairs;
  if (!pair && e >= q.experts) return;
  const int from = pair ? own : e << kPairBits, to = from + (1 << kPairBits);
  int ahead = 0, upto = 0;
#pragma unroll 2
  for (int j = 4 * part; j < pairs; j += 16) {
    const s32x4 v = *(const s32x4 *)(keys + j);
#pragma unroll
    for (int u = 0; u < 4; ++u) ahead += v[u] < from, upto += v[u] < to;
  }
#pragma unroll
  for (int o = 1; o <= 2; o <<= 1) ahead += __shfl_xor(ahead, o, 64), upto += __shfl_xor(upto, o, 64);   // (the four of an item together)
  if (pair) {
    if (part) return;
    const bool has = e < q.experts;
    q.place[item] = has ? ahead : -1;
    if (!has) return;
    q.tokens[ahead] = item / top;
    if (q.by_place) q.by_place[ahead] = weights[item];
    return;
  }
  const int count = upto - ahead, t0 = ahead / q.tile_m + e, t1 = e + 1 < q.experts ? upto / q.tile_m + e + 1 : q.max_tiles;
  for (int t = t0 + part; t < t1; t += 4) {
    const int first = (t - t0) * q.tile_m;
    q.tiles[3 * t] = first < count ? e : -1, q.tiles[3 * t + 1] = ahead + first, q.tiles[3 * t + 2] = min(q.tile_m, count - first);
  }
}

// A workgroup: TT tiles of 16 tokens.  Latencies: the inputs are split over the waves, every operand of U steps is asked for before the first is
// used (16 waves: all of 2048 inputs at once), and the choice of a token with up to 64 outputs stays in one wave's registers.  Few tokens: 16 waves
// share a tile, so that a wave chooses for one token; many: eight waves (mv_moe_route).  34 outputs of 2048 inputs, alone: 24 tokens 18.8 -> 11.0 us; one
// launch behind the other, eight waves with a step's loads at a time -> now: 24 tokens 14.7 -> 9.7, 9001 24 -> 16; 128 outputs of 512 inputs: one token
// 12.7 -> 12.8, 24 20.5 -> 15.4, 20000 53 -> 51; fp32, 34 outputs of 2048 inputs, 4400 tokens: 392 -> 131.  Now 9001 tokens with the choices of four tokens
// at once, one launch between events, 29.3 -> 24.4: 8.5 of 20 us are the products (their inputs by half lines), 282 workgroups on 256 CUs.
// GROUP (one workgroup has all tokens): the choices stay in LDS for the grouping behind them, a launch and a trip to memory less.  Both products with what is around them, 32
// experts: 12 tokens of 4 choices (2048 -> 768) 67.2 -> 65.7 us, 4 of 8 (1024 -> 384; the host's) 48.5 -> 44.5.  Up to one tile: two tiles in one
// workgroup in place of two workgroups cost more than the launch (24 of 4 70.2 -> 74.0, 32 of 8 84 -> 95).  Router, grouping and products in a graph, grouped by another
// launch and here, 16 experts of 512 -> 128: 64 pairs 15.2 and 12.4, 128 16.8 and 14.5, 192 18.3 and 16.6; 256 of 2048 -> 768, which would be on the other side of the line, 56.5 either way.
template <typename Tag, int WAVES, int TT, bool GROUP>
__global__ void __launch_bounds__(WAVES * 64) moe_route_kernel(RouteParams p, RouteGroups q) {
  typedef typename elem<Tag>::T T;
  static_assert(!GROUP || (WAVES == 16 && TT == 1 && !__is_same(Tag, f32_tag)), "sixteen waves group, in the place of the partial tiles");
  constexpr int TOKENS = 16 * TT, U = WAVES == 16 ? 4 : 2;
  extern __shared__ float lds[];   // logits [TOKENS][outputs] | scratch [TOKENS][outputs] | (16-bit) partial tiles
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), m0 = blockIdx.x * TOKENS, R = p.outputs;
  float *sc = lds, *ch = sc + TOKENS * R;
  const T *x = (const T *)p.x, *w = (const T *)p.w;
  constexpr bool FOUR = WAVES < TOKENS;
  float corrections[4] = {};   // (asked for ahead of the products)
  if (p.correction)
#pragma unroll
    for (int j = 0; j < (FOUR ? 4 : 1); ++j) corrections[j] = elem<Tag>::ld(((const T *)p.correction)[min(FOUR ? j * 16 + (lane & 15) : lane, R - 1)]);
  if constexpr (__is_same(Tag, f32_tag)) {
    const int l = tid & 15;
    for (int i = tid >> 4; i < TOKENS * R; i += WAVES * 4) {
      const int t = i / R, r = i - t * R;
      const T *xr = x + (int64_t)min(m0 + t, p.rows - 1) * p.x_stride, *wr = w + (int64_t)r * p.k;
      float z = 0.f;
      int k = l;
      for (; k < p.k - 112; k += 128) {   // (eight steps' loads in flight, one sum)
        float a[8], b[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) a[u] = xr[k + 16 * u], b[u] = wr[k + 16 * u];
#pragma unroll
        for (int u = 0; u < 8; ++u) z = fmaf(a[u], b[u], z);
      }
      for (; k < p.k; k += 16) z = fmaf(xr[k], wr[k], z);
      z = row16_sum(z);
      if (l == 0) sc[i] = z;
    }
  } else {
    f32x4 *part = (f32x4 *)(ch + TOKENS * R);   // [waves][kRouteTiles][TT][64]
    const int r16 = lane & 15, g = lane >> 4, steps = p.k / 32;
    const T *xr[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) xr[t] = x + (int64_t)min(m0 + t * 16 + r16, p.rows - 1) * p.x_stride + g * 8;
    for (int rt = 0; rt * 16 < R; rt += kRouteTiles) {
      const int tiles = min(kRouteTiles, (R + 15) / 16 - rt);
      auto products = [&](auto TILES) __attribute__((always_inline)) {   // a wave: a run of the inputs, so that it uses whole lines of the weights
        constexpr int NT = decltype(TILES)::value;
        const T *wr[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) wr[j] = w + (int64_t)min((rt + j) * 16 + r16, R - 1) * p.k + g * 8;
        f32x4 acc[NT][TT] = {};
        const int hi = steps * (wave + 1) / WAVES;
        for (int s = steps * wave / WAVES; s < hi; s += U) {
          u32x4 a[U][NT], b[U][TT];
#pragma unroll
          for (int u = 0; u < U; ++u)
            if (s + u < hi) {   // (of the wave: few inputs are not asked for several times)
              const int at = (s + u) * 32;
#pragma unroll
              for (int t = 0; t < TT; ++t) b[u][t] = *(const u32x4 *)(xr[t] + at);
#pragma unroll
              for (int j = 0; j < NT; ++j) a[u][j] = *(const u32x4 *)(wr[j] + at);
            }
#pragma unroll
          for (int u = 0; u < U; ++u)
            if (s + u < hi) {
#pragma unroll
              for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int t = 0; t < TT; ++t) acc[j][t] = mfma16x16x32<Tag>(a[u][j], b[u][t], acc[j][t]);
            }
        }
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int t = 0; t < TT; ++t) part[((wave * kRouteTiles + j) * TT + t) * 64 + lane] = acc[j][t];
      };
      if (tiles == 1) products(std::integral_constant<int, 1>{});
      else if (tiles == 2) products(std::integral_constant<int, 2>{});
      else if (tiles == 3) products(std::integral_constant<int, 3>{});
      else products(std::integral_constant<int, 4>{});
      __syncthreads();
      for (int i = wave; i < tiles * TT; i += WAVES) {
        const int j = i / TT, t = i - j * TT;
        f32x4 z = part[(j * TT + t) * 64 + lane];
#pragma unroll
        for (int v = 1; v < WAVES; ++v) z += part[((v * kRouteTiles + j) * TT + t) * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = (rt + j) * 16 + g * 4 + e;
          if (r < R) sc[(t * 16 + r16) * R + r] = z[e];
        }
      }
      __syncthreads();
    }
  }
  int *keys = GROUP ? (int *)(ch + TOKENS * R) : nullptr;
  float *weights_too = GROUP ? (float *)(keys + kRouteItems + 16) : nullptr;
  __syncthreads();
  if constexpr (GROUP) {
    if (tid < 16) keys[p.rows * p.top + tid] = INT32_MAX;
  }
  if (FOUR && R <= 64 && p.groups <= 8) {
    for (int t = wave * 4 + (lane >> 4); t < TOKENS; t += WAVES * 4) choose_four<Tag>(p, sc + t * R, m0 + t, m0 + t < p.rows, corrections);
    return;
  }
  for (int t = wave; t < TOKENS && m0 + t < p.rows; t += WAVES) choose<Tag>(p, sc + t * R, ch + t * R, m0 + t, corrections[0], keys, weights_too);   // (no barrier in it)
  if constexpr (GROUP) {
    __syncthreads();
    group_few(q, keys, weights_too, p.rows * p.top, p.top);
  }
}

// ---- grouping.  Workgroup (e, part): the pairs of expert e, which start behind those of the experts before it.  Each wave walks a run of all
// pairs, in order, so places are the same in every run: all of its run to count, then the part of it whose pairs it places.  Latencies and the stores
// to scattered places bound it, and instructions that are fetched for the first time: all of a run's choices at once, kept in registers for the second
// walk, made a program that took longer to arrive than the second reading (36004 pairs, eight parts 25.6 us).  36004 pairs of 32 experts: one part
// 17.4 us, eight 10.1; 160000 pairs 61.6 and 27.8; 4000 pairs 5.9 and 5.9.
constexpr int kGroupThreads = 1024, kGroupWaves = kGroupThreads / 64, kGroupAhead = 8;   // kGroupAhead: choices of a lane requested at a time
constexpr int kGroupParts = 8;

__global__ void __launch_bounds__(kGroupThreads) moe_group_kernel(const int32_t *ids, int pairs, int top, int experts, int tile_m,
                                                                  int max_tiles, int32_t *rows, int32_t *tokens, int32_t *tiles,
                                                                  const float *weights, float *weights_out) {
  __shared__ int less[kGroupWaves], equal[kGroupWaves];
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int runs = (pairs + kGroupWaves * 64 - 1) / (kGroupWaves * 64), lo = wave * runs * 64, hi = min(pairs, lo + runs * 64);
  // the pairs of its run that the wave places: from `from` on, ahead of `to`
  const int parts = gridDim.y, part = blockIdx.y;
  int from = lo, to = hi;
  if (parts > 1) from = lo + runs * part / parts * 64, to = min(hi, lo + runs * (part + 1) / parts * 64);
  int nl = 0, ne = 0, nb = 0;   // choices of lower experts, of this one, of this one ahead of `from`
  // the choices i0 + 64 u + lane, ahead of `end` (-1 behind it)
  auto choices = [&](int i0, int end, int (&v)[kGroupAhead]) {
#pragma unroll
    for (int u = 0; u < kGroupAhead; ++u) {
      const int i = i0 + 64 * u + lane;
      v[u] = ids[min(i, pairs - 1)];
      if (i >= end) v[u] = -1;
    }
  };
  for (int i0 = lo; i0 < hi; i0 += 64 * kGroupAhead) {
    int v[kGroupAhead];
    choices(i0, hi, v);
#pragma unroll
    for (int u = 0; u < kGroupAhead; ++u) {
      const int is = v[u] == e;
      nl += v[u] >= 0 && v[u] < e, ne += is, nb += i0 + 64 * u < from ? is : 0;
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) nl += __shfl_xor(nl, o, 64), ne += __shfl_xor(ne, o, 64);
  if (part) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) nb += __shfl_xor(nb, o, 64);
  }
  if (lane == 0) less[wave] = nl, equal[wave] = ne;
  __syncthreads();
  int start = 0, count = 0, ahead = nb;
  for (int w = 0; w < kGroupWaves; ++w) {
    start += less[w], count += equal[w];
    if (w < wave) ahead += equal[w];
  }
  int at = start + ahead;
  for (int i0 = from; i0 < to; i0 += 64 * kGroupAhead) {
    int v[kGroupAhead];
    float w[kGroupAhead];
    choices(i0, to, v);
#pragma unroll
    for (int u = 0; u < kGroupAhead; ++u)
      if (weights && v[u] == e) w[u] = weights[i0 + 64 * u + lane];
#pragma unroll
    for (int u = 0; u < kGroupAhead; ++u) {
      const int i = i0 + 64 * u + lane;
      const unsigned long long mask = __ballot(v[u] == e);
      if (v[u] == e) {
        const int place = at + __popcll(mask & ((1ull << lane) - 1));
        rows[i] = place, tokens[place] = i / top;
        if (weights) weights_out[place] = w[u];
      }
      if (e == 0 && v[u] >= experts) rows[i] = -1;
      at += __popcll(mask);
    }
  }
  if (part) return;
  // tiles of this expert: entries start / tile_m + e on, up to the next expert's; the last expert also clears what is left
  const int t0 = start / tile_m + e, t1 = e + 1 < experts ? (start + count) / tile_m + e + 1 : max_tiles;
  for (int t = t0 + tid; t < t1; t += kGroupThreads) {
    const int first = (t - t0) * tile_m;
    tiles[3 * t] = first < count ? e : -1, tiles[3 * t + 1] = start + first, tiles[3 * t + 2] = min(tile_m, count - first);
  }
}

// ---- products over the groups ---------------------------------------------------------------------------------------------
struct MoeLinear {
  const void *x, *w;
  void *out;
  const int32_t *tokens, *tiles;   // tokens NULL: row = place
  const float *in_scale;           // by place; NULL: 1
  int64_t x_stride, out_stride, w_expert;   // w_expert: elements between two experts' weights
  int n, k;                        // outputs (gated: of the product with up), inputs
  MvGateAct act;
};

__device__ __forceinline__ float in_scale_of(const MoeLinear &p, int place) { return p.in_scale ? p.in_scale[place] : 1.0f; }

// few rows per expert: TM tiles of 16 rows, TN of 16 outputs; the waves split the inputs, weight fragments come straight from
// memory in the order they are stored (1 KiB per instruction)
template <typename Tag, int TM, int TN, bool GATED>
__global__ void __launch_bounds__(256) moe_small_kernel(MoeLinear p) {
  typedef typename elem<Tag>::T T;
  constexpr int NA = GATED ? 2 * TN : TN, U = NA + TM >= 6 ? 2 : 4;
  __shared__ f32x4 red[4][NA * TM][64];
  const int32_t *tile = p.tiles + 3 * blockIdx.y;
  const int e = tile[0], m0 = tile[1], live = tile[2];
  if (e < 0) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r16 = lane & 15, g = lane >> 4;
  const int steps = p.k / 32, s_lo = steps * wave / 4, s_hi = steps * (wave + 1) / 4, ntiles = p.n / 16;
  const u32x4 *w[NA];
#pragma unroll
  for (int j = 0; j < NA; ++j) {
    const int t = min((int)blockIdx.x * TN + (GATED ? j >> 1 : j), ntiles - 1) + (GATED && (j & 1) ? ntiles : 0);
    w[j] = (const u32x4 *)((const T *)p.w + e * p.w_expert) + (int64_t)t * steps * 64 + lane;
  }
  const T *x[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int place = m0 + min(i * 16 + r16, live - 1);
    x[i] = (const T *)p.x + (int64_t)(p.tokens ? p.tokens[place] : place) * p.x_stride + g * 8;
  }
  f32x4 acc[NA][TM] = {};
  for (int s = s_lo; s < s_hi; s += U) {
    u32x4 a[U][NA], b[U][TM];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(s + u, s_hi - 1);
#pragma unroll
      for (int j = 0; j < NA; ++j) a[u][j] = __builtin_nontemporal_load(w[j] + k * 64);
#pragma unroll
      for (int i = 0; i < TM; ++i) b[u][i] = *(const u32x4 *)(x[i] + k * 32);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s + u < s_hi) {
#pragma unroll
        for (int j = 0; j < NA; ++j)
#pragma unroll
          for (int i = 0; i < TM; ++i) acc[j][i] = mfma16x16x32<Tag>(a[u][j], b[u][i], acc[j][i]);
      }
  }
#pragma unroll
  for (int j = 0; j < NA; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) red[wave][j * TM + i][lane] = acc[j][i];
  __syncthreads();
  auto total = [&](int t) { return (red[0][t][lane] + red[1][t][lane]) + (red[2][t][lane] + red[3][t][lane]); };
  for (int t = wave; t < TN * TM; t += 4) {
    const int j = t / TM, i = t - j * TM, row = i * 16 + r16, n0 = ((int)blockIdx.x * TN + j) * 16;
    if (row >= live || n0 >= p.n) continue;
    const float sc = in_scale_of(p, m0 + row);
    f32x4 o;
    if constexpr (GATED) {
      const f32x4 gate = total(2 * j * TM + i) * sc, up = total((2 * j + 1) * TM + i) * sc;
#pragma unroll
      for (int q = 0; q < 4; ++q) o[q] = gated_act<Tag>(gate[q], up[q], p.act);
    } else {
      o = total(t) * sc;
    }
    *(u32x2 *)((T *)p.out + (int64_t)(m0 + row) * p.out_stride + n0 + g * 4) = pack_quad<Tag>(o);
  }
}

// A fragment of 16 rows x 32 inputs that LDS-DMA brings: four adjacent lanes fetch one row's 64 bytes (16 rows in adjacent lanes would be
// 16 cache lines), in an order that spreads the rows' like pieces over the banks.
__device__ __forceinline__ int row_chunk(int lane) { return (lane & 3) ^ ((lane >> 4) & 3); }              // the piece that a lane fetches
__device__ __forceinline__ int row_place(int row, int chunk) { return row * 4 + (chunk ^ ((row >> 2) & 3)); }  // where a piece lies

// many rows: BM x BN per workgroup of 2 x 2 waves, 64 inputs at a time.  Rows and weights reach LDS by DMA as fragments (16 rows x
// 32 inputs, 1 KiB; weights in the order of the lanes); the next 64 inputs land while these are multiplied.
// QUARTERS: sums as moe_small_kernel makes them, of four quarters of the inputs, so that an expert of some 30 rows gives the same bits from either.
template <typename Tag, int BM, int BN, bool GATED, bool QUARTERS>
__global__ void __launch_bounds__(256, 2) moe_tile_kernel(MoeLinear p) {
  typedef typename elem<Tag>::T T;
  constexpr int MT = BM / 16, NT = BN / 16, WM = MT / 2, WN = NT / 2, PIECES = 2 * (MT + NT), PER = PIECES / 4;
  constexpr int STAGE = PIECES * 1024;
  extern __shared__ __attribute__((aligned(16))) char smem[];   // 2 stages of [rows: MT][2] | [weights: NT][2] fragments
  const int32_t *tile = p.tiles + 3 * blockIdx.y;
  const int e = tile[0], m0 = tile[1], live = tile[2];
  if (e < 0) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4;
  const int wm = wave & 1, wn = wave >> 1, ntiles = p.n / 16, steps = p.k / 32, nt0 = blockIdx.x * (GATED ? NT / 2 : NT);
  // this wave's pieces: piece = i * 4 + wave = (tile, half of the 64 inputs); a piece's address moves by a constant per trip
  const T *src[PER];
  int64_t step[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int piece = i * 4 + wave, half = piece & 1, t = piece >> 1;
    if (t < MT) {
      const int place = m0 + min(t * 16 + (lane >> 2), live - 1);
      src[i] = (const T *)p.x + (int64_t)(p.tokens ? p.tokens[place] : place) * p.x_stride + half * 32 + row_chunk(lane) * 8;
      step[i] = 64;
    } else {
      const int j = t - MT, wt = min(nt0 + (GATED ? j >> 1 : j), ntiles - 1) + (GATED && (j & 1) ? ntiles : 0);
      src[i] = (const T *)p.w + e * p.w_expert + ((int64_t)wt * steps + half) * 512 + lane * 8;
      step[i] = 1024;
    }
  }
  auto fetch = [&](int buf) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src[i],
                                       (__attribute__((address_space(3))) void *)(smem + buf * STAGE + (i * 4 + wave) * 1024), 16, 0, 0);
      src[i] += step[i];
    }
  };
  f32x4 acc[WN][WM] = {};
  const uint32_t base = lds_address(smem) + lane * 16, rows = lds_address(smem) + row_place(r16, g) * 16;
  const int trips = p.k / 64;
  f32x4 half[2][WN][WM] = {};   // (of the first two quarters, of the third)
  int quarter = 0;
  auto settle = [&](int done) {   // the quarters that end behind `done` steps of 32 inputs
    while (quarter < 3 && steps * (quarter + 1) / 4 == done) {
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int i = 0; i < WM; ++i) {
          if (quarter == 2) half[1][j][i] = acc[j][i];
          else if (quarter == 1) half[0][j][i] += acc[j][i];
          else half[0][j][i] = acc[j][i];
          acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      ++quarter;
    }
  };
  if constexpr (QUARTERS) settle(0);
  fetch(0);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  lds_barrier();
  for (int t = 0; t < trips; ++t) {
    if (t + 1 < trips) fetch((t + 1) & 1);
    const uint32_t at = (t & 1) * STAGE, xa = rows + at + wm * WM * 2048, wa = base + at + (MT + wn * WN) * 2048;
    u32x4 a[2][WN], b[2][WM];
    static_for<2>([&](auto H) {
      constexpr int h = decltype(H)::value;
      static_for<WM>([&](auto I) { lds_read128<decltype(I)::value * 2048 + h * 1024>(b[h][decltype(I)::value], xa); });
      static_for<WN>([&](auto I) { lds_read128<decltype(I)::value * 2048 + h * 1024>(a[h][decltype(I)::value], wa); });
    });
    static_for<2>([&](auto H) {
      constexpr int h = decltype(H)::value;
      static_for<WM>([&](auto I) { lds_wait<h == 0 ? WM + WN : 0>(b[h][decltype(I)::value]); });
      static_for<WN>([&](auto I) { lds_wait<h == 0 ? WM + WN : 0>(a[h][decltype(I)::value]); });
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int i = 0; i < WM; ++i) acc[j][i] = mfma16x16x32<Tag>(a[h][j], b[h][i], acc[j][i]);
      if constexpr (QUARTERS) settle(2 * t + h + 1);
    });
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
  }
  if constexpr (QUARTERS) {
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int i = 0; i < WM; ++i) acc[j][i] = half[0][j][i] + (half[1][j][i] + acc[j][i]);
  }
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int row = (wm * WM + i) * 16 + r16;
    if (row >= live) continue;
    const float sc = in_scale_of(p, m0 + row);
    T *out = (T *)p.out + (int64_t)(m0 + row) * p.out_stride + g * 4;
#pragma unroll
    for (int j = 0; j < (GATED ? WN / 2 : WN); ++j) {
      const int nt = nt0 + (GATED ? wn * (WN / 2) + j : wn * WN + j);
      if (nt >= ntiles) continue;
      f32x4 o;
      if constexpr (GATED) {
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = gated_act<Tag>(acc[2 * j][i][q] * sc, acc[2 * j + 1][i][q] * sc, p.act);
      } else {
        o = acc[j][i] * sc;
      }
      *(u32x2 *)(out + nt * 16) = pack_quad<Tag>(o);
    }
  }
}

// Very many rows: 128 x 256 per workgroup of four waves side by side, two workgroups to a CU, so that one multiplies while the other starts or ends.
// Bound by the matrix cores and their power, if the operands are there in time: three stages of 32 inputs, of which two are under way, and the operands of a stage
// are read one by one between the products of the stage before, as are the next transfers asked for.  A stage takes 1224 cycles where its products are 1024 (two
// workgroups) and those with their transfers alone 1084, at 1.65 of 2.4 GHz.  And by rounds: 9001 tokens of
// 4 choices are 1728 gated and 2304 plain workgroups (2048 -> 2 x 768, 768 -> 2048) on 512 places, 3.4 and 4.5 rounds.  Rows come 64 inputs at a time, in whole lines of memory, every other stage.
// Results leave through LDS, 128 bytes of a row (gated: 64) to a store.
// Workgroups are dealt to the XCDs in turn, and each XCD gets a run of an eighth of the work (eight tiles of rows and all their outputs at a time, the
// rows first): its L2 holds what its workgroups share, and none has more than the others.
// 36004 pairs of 32 experts, 2048 -> 2 x 768 gated and 768 -> 2048: 343 + 198 us (one workgroup of 256 x 256 to a CU, two stages of 64 inputs, four
// tiles to an XCD in turn) -> 260 + 157 (rows by half lines, transfers at the start of a stage, tiles looked for one trip to memory behind the other; the layer
// with all that is beside them 483) -> the layer 449 (460 where 512 tiles are always asked for: the search 2.7 us of a workgroup's 65 -> 1.6).
constexpr int kWideRows = 128, kWideStages = 3;
// place of a row's piece among its eight, and the piece at a place: the lanes of a read (four each of different rows) are at different banks
__device__ __forceinline__ int wide_piece(int row, int piece) { return piece ^ (row >> 1 & 7); }
template <typename Tag, bool GATED, int ACT>
__device__ __forceinline__ float wide_result(float x, float up, MvGateAct act) {
  if constexpr (!GATED) return x;
  act.kind = ACT;   // (known at compile time: one branch per workgroup, not per output)
  return gated_act<Tag>(x, up, act);
}

template <typename Tag, bool GATED>
__global__ void __launch_bounds__(256, 2) moe_wide_kernel(MoeLinear p, int nx, int max_tiles) {
  typedef typename elem<Tag>::T T;
  constexpr int TILES = 16, WM = 8, WN = 4, WSTAGE = TILES * 1024, XSTAGE = WM * 2048;
  extern __shared__ __attribute__((aligned(16))) char smem[];   // three stages of weights, two of rows (64 inputs)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4;
  // the halves of a tile of 256 rows that are there: tiles 64 c + lane, all that there may be asked for at once (more than 512: once more for
  // the one that is looked for)
  constexpr int AHEAD = 8;
  int info[AHEAD][3];
  auto look = [&](int i0) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < AHEAD; ++c)
      if (c == 0 || i0 + 64 * c < max_tiles)
#pragma unroll
        for (int q = 0; q < 3; ++q) info[c][q] = p.tiles[3 * min(i0 + 64 * c + lane, max_tiles - 1) + q];
  };
  auto upper_of = [&](int c, int i0) { return __ballot(i0 + 64 * c + lane < max_tiles && info[c][0] >= 0); };
  auto lower_of = [&](int c, int i0) { return __ballot(i0 + 64 * c + lane < max_tiles && info[c][0] >= 0 && info[c][2] > kWideRows); };
  int total = 0, held = 0;
  for (int i0 = 0; i0 < max_tiles; i0 += 64 * AHEAD) {
    look(held = i0);
#pragma unroll
    for (int c = 0; c < AHEAD; ++c)
      if (c == 0 || i0 + 64 * c < max_tiles) total += __popcll(upper_of(c, i0)) + __popcll(lower_of(c, i0));
  }
  const int per = (total * nx + 7) / 8, turn = blockIdx.x >> 3, index = (blockIdx.x & 7) * per + turn;
  if (turn >= per || index >= total * nx) return;
  const int group = index / (8 * nx), in = index - group * 8 * nx, high = min(8, total - group * 8), tx = in / high;
  int nth = group * 8 + in % high, e = -1, m0 = 0, live = 0;
  for (int i0 = 0; e < 0; i0 += 64 * AHEAD) {
    if (i0 != held) look(held = i0);
#pragma unroll
    for (int c = 0; c < AHEAD; ++c) {
      if (nth < 0) break;
      const unsigned long long upper = upper_of(c, i0), lower = lower_of(c, i0);
      const int n = __popcll(upper) + __popcll(lower);
      if (nth < n) {
        const unsigned long long below = (1ull << lane) - 1;
        const int ahead = __popcll(upper & below) + __popcll(lower & below);
        const bool second = (lower >> lane & 1) && nth == ahead + 1;
        const int mine = __ffsll(__ballot((upper >> lane & 1) && (nth == ahead || second))) - 1, skip = __ballot(second) ? kWideRows : 0;
        e = __builtin_amdgcn_readlane(info[c][0], mine), m0 = __builtin_amdgcn_readlane(info[c][1], mine) + skip;
        live = __builtin_amdgcn_readlane(info[c][2], mine) - skip;
      }
      nth -= n;
    }
  }
  const int ntiles = p.n / 16, steps = p.k / 32, nt0 = tx * (GATED ? TILES / 2 : TILES);
  // this wave's transfers: eight rows x 64 inputs (whole lines of memory), of which there are four to a wave every other stage; four fragments of weights
  const T *xs[4], *ws[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int j = 4 * i + wave, wt = min(nt0 + (GATED ? j >> 1 : j), ntiles - 1) + (GATED && (j & 1) ? ntiles : 0);
    ws[i] = (const T *)p.w + e * p.w_expert + (int64_t)wt * steps * 512;
    const int row = j * 8 + (lane >> 3), place = m0 + min(row, live - 1);
    xs[i] = (const T *)p.x + (int64_t)(p.tokens ? p.tokens[place] : place) * p.x_stride + (wide_piece(row & 15, lane & 7)) * 8;
  }
  const int lane8 = lane * 8;
  auto transfer = [&](const T *from, char *to) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)from, (__attribute__((address_space(3))) void *)to, 16, 0, 0);
  };
  auto fetch_w = [&](int i, int t, int slot) __attribute__((always_inline)) { transfer(ws[i] + (int64_t)t * 512 + lane8, smem + slot * WSTAGE + (4 * i + wave) * 1024); };
  auto fetch_x = [&](int i, int u) __attribute__((always_inline)) { transfer(xs[i] + (int64_t)u * 64, smem + kWideStages * WSTAGE + (u & 1) * XSTAGE + (4 * i + wave) * 1024); };
  // stages 0 .. 2 of the weights, 0 .. 3 of the rows, in the order in which they are needed
  for (int t = 0; t < min(kWideStages, steps); ++t) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (t != 1) fetch_x(i, t >> 1);
      fetch_w(i, t, t);
    }
  }
  f32x4 acc[WN][WM] = {};
  const uint32_t rows = lds_address(smem) + kWideStages * WSTAGE + r16 * 128, weights = lds_address(smem) + lane * 16 + wave * WN * 1024;
  const int piece_of[2] = {wide_piece(r16, g) * 16, wide_piece(r16, 4 + g) * 16};
  u32x4 a[2][WN], b[2][WM];
  auto landed = [&](auto H) __attribute__((always_inline)) {
    constexpr int h = decltype(H)::value;
    static_for<WN>([&](auto I) { lds_wait<0>(a[h][decltype(I)::value]); });
    static_for<WM>([&](auto I) { lds_wait<0>(b[h][decltype(I)::value]); });
  };
  int slot = 0;
  auto step = [&](auto H, int t) __attribute__((always_inline)) {
    constexpr int h = decltype(H)::value;
    // stage t + 1 is there, and every wave has stage t in registers, whose place the stage three ahead takes (rows: that of stages t - 1 and t, at odd t)
    if (t + kWideStages - 1 < steps) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(h == 0 ? 8 : 4) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    const bool ahead = t + kWideStages < steps;
    const int free = slot;
    slot = slot == kWideStages - 1 ? 0 : slot + 1;
    // (behind the last stage: an old one, for nobody)
    const uint32_t xa = rows + (h ? ((t + 1) >> 1 & 1) : (t >> 1 & 1)) * XSTAGE + piece_of[1 - h], wa = weights + slot * WSTAGE;
    static_for<WM>([&](auto I) {
      constexpr int i = decltype(I)::value;
      if constexpr (i < WN) lds_read128<i * 1024>(a[1 - h][i], wa);
      lds_read128<i * 2048>(b[1 - h][i], xa);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < WN; ++j) acc[j][i] = mfma16x16x32<Tag>(a[h][j], b[h][i], acc[j][i]);
      if (ahead) {
        if constexpr (i >= 4) fetch_w(i - 4, t + kWideStages, free);
        else if constexpr (h == 1) fetch_x(i, (t + kWideStages) >> 1);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    landed(std::integral_constant<int, 1 - h>{});
  };
  if (steps >= kWideStages) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  lds_barrier();
  static_for<WN>([&](auto I) { lds_read128<decltype(I)::value * 1024>(a[0][decltype(I)::value], weights); });
  static_for<WM>([&](auto I) { lds_read128<decltype(I)::value * 2048>(b[0][decltype(I)::value], rows + piece_of[0]); });
  landed(std::integral_constant<int, 0>{});
  for (int t = 0; t < steps; t += 2) {   // (an even number of them)
    step(std::integral_constant<int, 0>{}, t);
    step(std::integral_constant<int, 1>{}, t + 1);
  }
  // (every wave has its last stage in registers, and no transfer is under way: LDS is free)
  float sc[WM];
#pragma unroll
  for (int i = 0; i < WM; ++i) sc[i] = in_scale_of(p, m0 + min(i * 16 + r16, live - 1));
  constexpr int COLS = GATED ? WN * 8 : WN * 16, ROW = COLS * 2 + 16, PIECES = COLS / 8;   // outputs of a wave; bytes of a row of them, 16-byte pieces
  char *const mine_at = smem + wave * (kWideRows * ROW);
  const int first = nt0 * 16 + wave * COLS;
  auto results = [&](auto A) {
    constexpr int ACT = decltype(A)::value;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < COLS / 16; ++j) {
        f32x4 o;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          o[q] = GATED ? wide_result<Tag, true, ACT>(acc[GATED ? 2 * j : j][i][q] * sc[i], acc[GATED ? 2 * j + 1 : j][i][q] * sc[i], p.act)
                       : acc[j][i][q] * sc[i];
        *(u32x2 *)(mine_at + (i * 16 + r16) * ROW + j * 32 + g * 8) = pack_quad<Tag>(o);
      }
  };
  if (!GATED) results(std::integral_constant<int, 0>{});
  else if (p.act.kind == MV_ACT_GELU) results(std::integral_constant<int, MV_ACT_GELU>{});
  else if (p.act.kind == MV_ACT_CLAMPED) results(std::integral_constant<int, MV_ACT_CLAMPED>{});
  else if (p.act.kind == MV_ACT_RELU) results(std::integral_constant<int, MV_ACT_RELU>{});
  else results(std::integral_constant<int, MV_ACT_SILU>{});
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  const int piece = lane % PIECES, col = first + piece * 8;
#pragma unroll
  for (int n = 0; n < kWideRows * PIECES / 64; ++n) {
    const int row = n * (64 / PIECES) + lane / PIECES;
    const u32x4 v = *(const u32x4 *)(mine_at + row * ROW + piece * 16);
    if (row < live && col < p.n) *(u32x4 *)((T *)p.out + (int64_t)(m0 + row) * p.out_stride + col) = v;
  }
}

// fp32: 16 rows x 64 outputs per workgroup, weights [expert][outputs (gate | up)][inputs]
template <bool GATED>
__global__ void __launch_bounds__(256) moe_f32_kernel(MoeLinear p) {
  constexpr int K = 32, NW = GATED ? 128 : 64;
  __shared__ float xs[16][K + 1], ws[NW][K + 1];
  const int32_t *tile = p.tiles + 3 * blockIdx.y;
  const int e = tile[0], m0 = tile[1], live = tile[2], tid = threadIdx.x, n0 = blockIdx.x * 64;
  if (e < 0) return;
  const float *w = (const float *)p.w + e * p.w_expert;
  const int c = tid & 63, r = tid >> 6;   // column; rows r, r + 4, ...
  float acc[4] = {}, up[4] = {};
  for (int k0 = 0; k0 < p.k; k0 += K) {
    __syncthreads();
    for (int i = tid; i < 16 * K; i += 256) {
      const int t = i / K, k = i - t * K, place = m0 + min(t, live - 1);
      xs[t][k] = ((const float *)p.x)[(int64_t)(p.tokens ? p.tokens[place] : place) * p.x_stride + k0 + k];
    }
    for (int i = tid; i < NW * K; i += 256) {
      const int j = i / K, k = i - j * K, n = min(n0 + (j & 63), p.n - 1) + (j >= 64 ? p.n : 0);
      ws[j][k] = w[(int64_t)n * p.k + k0 + k];
    }
    __syncthreads();
    for (int k = 0; k < K; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[i] = fmaf(xs[r + 4 * i][k], ws[c][k], acc[i]);
        if constexpr (GATED) up[i] = fmaf(xs[r + 4 * i][k], ws[64 + c][k], up[i]);
      }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (r + 4 * i < live && n0 + c < p.n) {
      const float sc = in_scale_of(p, m0 + r + 4 * i);
      ((float *)p.out)[(int64_t)(m0 + r + 4 * i) * p.out_stride + n0 + c] = GATED ? gated_act<f32_tag>(acc[i] * sc, up[i] * sc, p.act) : acc[i] * sc;
    }
}

template <typename Tag, bool GATED>
int launch_linear(const MoeLinear &p, int tile_m, int max_tiles, hipStream_t st) {
  const int nt = p.n / 16;
  constexpr int TN = GATED ? 1 : 2;
  const dim3 small((nt + TN - 1) / TN, max_tiles);
  const bool quarters = tile_m & MV_MOE_QUARTERS;
  tile_m &= ~MV_MOE_QUARTERS;
  if (tile_m == 16) hipLaunchKernelGGL((moe_small_kernel<Tag, 1, TN, GATED>), small, dim3(256), 0, st, p);
  else if (tile_m == 32) hipLaunchKernelGGL((moe_small_kernel<Tag, 2, TN, GATED>), small, dim3(256), 0, st, p);
  else if (tile_m == 64) {
    constexpr int BN = 128;
    const dim3 grid((nt * 16 * (GATED ? 2 : 1) + BN - 1) / BN, max_tiles);
    if (quarters) hipLaunchKernelGGL((moe_tile_kernel<Tag, 64, BN, GATED, true>), grid, dim3(256), (64 + BN) * 256, st, p);
    else hipLaunchKernelGGL((moe_tile_kernel<Tag, 64, BN, GATED, false>), grid, dim3(256), (64 + BN) * 256, st, p);
  } else if ((tile_m == 128 || tile_m == 256) && !quarters) {   // (tiles of 128 rows have one half)
    const int nx = (nt * (GATED ? 2 : 1) + 15) / 16;
    if (int rc = mv_allow_lds<moe_wide_kernel<Tag, GATED>>()) return rc;
    hipLaunchKernelGGL((moe_wide_kernel<Tag, GATED>), dim3((unsigned)(((int64_t)max_tiles * 2 * nx + 7) / 8 * 8)), dim3(256),
                       80 * 1024, st, p, nx, max_tiles);
  } else {
    return MV_E_SHAPE;
  }
  MV_LAUNCH_CHECK();
  return MV_OK;
}

template <typename Tag, int WAVES, int TT, bool GROUP = false>
int launch_route(const RouteParams &p, hipStream_t st, const RouteGroups &q = {}) {
  const size_t lds = (size_t)2 * 16 * TT * p.outputs * 4 + (__is_same(Tag, f32_tag) ? 0 : WAVES * kRouteTiles * TT * 1024);
  if (int rc = mv_allow_lds<moe_route_kernel<Tag, WAVES, TT, GROUP>>()) return rc;
  hipLaunchKernelGGL((moe_route_kernel<Tag, WAVES, TT, GROUP>), dim3((p.rows + 16 * TT - 1) / (16 * TT)), dim3(WAVES * 64), lds, st, p, q);
  return MV_OK;
}

}  // namespace

// `group` (or NULL): grouping along, where one workgroup has all tokens; *grouped says whether
static int route(const void *x, int64_t x_stride, const void *w, const void *correction, int32_t *ids, float *weights, int rows, int k, int outputs, int top, int groups,
                 int keep, float scale, int flags, int dtype, void *stream, const RouteGroups *group, bool *grouped) {
  if (rows == 0) return MV_OK;
  if (!x || !w || !ids || !weights) return MV_E_NULLPTR;
  if (flags & ~(MV_ROUTE_SIGMOID | MV_ROUTE_RAW)) return MV_E_RANGE;
  if (rows < 0 || k <= 0 || (k & 31) || outputs <= 0 || outputs > 512 || top <= 0 || top > 64 || top > outputs || groups <= 0 ||
      groups > 64 || outputs % groups || keep <= 0 || keep > groups || (int64_t)outputs / groups * keep < top || x_stride < k)
    return MV_E_SHAPE;
  if (!mv_aligned16(x) || !mv_aligned16(w) || x_stride % (dtype == MV_F32 ? 4 : 8)) return MV_E_ALIGN;
  const RouteParams p{x, w, correction, ids, weights, x_stride, rows, k, outputs, top, groups, keep, flags, scale};
  // A tile of 16 tokens over 16 waves while that fills no more than the chip.  More tokens: eight waves, so that the workgroups of a CU choose beside
  // each other (20000 tokens of 512 inputs, 128 outputs: 51 us, 16 waves 74, eight waves of two tiles 105; 384 outputs, whose scores leave room for one
  // workgroup a CU, 16 waves 123, eight 91).  Two tiles, which read the weights once, where those are long: 34 outputs of 4096 inputs, 4400 tokens
  // 23 us, one tile 28.  More than 64 outputs leave two tiles one workgroup a CU, so its rounds over the chip have to be full: 128 outputs of 4096
  // inputs, 4400 tokens 73 us, 12000 145; one tile 87 and 122.  LDS has the scores of two tiles up to 256 outputs.
  const bool along = group && dtype != MV_F32 && rows <= kRouteRows && rows * top + group->experts <= kRouteItems && outputs <= 64 && groups <= 8;
  MV_DISPATCH_DTYPE(dtype, {
    const hipStream_t st = (hipStream_t)stream;
    const bool full = k > 2048 && (rows <= 8192 || (k >= 4096 && (rows - 1) % 8192 >= 4096));
    int rc = MV_E_DTYPE;
    if (along) {
      if constexpr (!__is_same(Tag, f32_tag)) rc = launch_route<Tag, 16, 1, true>(p, st, *group);
    } else if (rows <= 16 * 256) rc = launch_route<Tag, 16, 1>(p, st);
    else if (dtype != MV_F32 && (outputs <= 64 ? k >= 2048 : outputs <= 256 && full)) rc = launch_route<Tag, 8, 2>(p, st);
    else rc = launch_route<Tag, 8, 1>(p, st);
    if (rc) return rc;
  });
  MV_LAUNCH_CHECK();
  if (along) *grouped = true;
  return MV_OK;
}

extern "C" int mv_moe_route(const void *x, int64_t x_stride, const void *w, const void *correction, int32_t *ids, float *weights,
                            int rows, int k, int outputs, int top, int groups, int keep, float scale, int flags, int dtype, void *stream) {
  return route(x, x_stride, w, correction, ids, weights, rows, k, outputs, top, groups, keep, scale, flags, dtype, stream, nullptr, nullptr);
}

extern "C" int mv_moe_group(const int32_t *ids, int pairs, int top, int experts, int tile_m, int max_tiles, int32_t *rows,
                            int32_t *tokens, int32_t *tiles, const float *weights, float *weights_out, void *stream) {
  if (pairs == 0) return MV_OK;
  if (!ids || !rows || !tokens || !tiles || (weights && !weights_out)) return MV_E_NULLPTR;
  if (pairs < 0 || top <= 0 || experts <= 0 || experts > 65535 || tile_m <= 0 || max_tiles < pairs / tile_m + experts) return MV_E_SHAPE;
  // (every part counts all pairs; a part is worth having for some 1024 of them to place)
  const int parts = std::max(1, std::min({kGroupParts, 256 / experts, pairs / 1024}));
  hipLaunchKernelGGL(moe_group_kernel, dim3(experts, parts), dim3(kGroupThreads), 0, (hipStream_t)stream, ids, pairs, top, experts, tile_m,
                     max_tiles, rows, tokens, tiles, weights, weights_out);
  MV_LAUNCH_CHECK();
  return MV_OK;
}

extern "C" int mv_moe_linear(const MvMoeLinearArgs *a, int dtype, void *stream) {
  if (!a || !a->x || !a->w || !a->out || !a->tiles) return MV_E_NULLPTR;
  if (dtype != MV_BF16 && dtype != MV_F16 && dtype != MV_F32) return MV_E_DTYPE;
  if (a->max_tiles <= 0) return a->max_tiles == 0 ? MV_OK : MV_E_SHAPE;
  if (a->max_tiles > 65535 || a->n <= 0 || a->k <= 0 || (a->k & 63) || (a->n & 15) || a->x_stride < a->k || a->out_stride < a->n)
    return MV_E_SHAPE;
  const int vec = dtype == MV_F32 ? 4 : 8;
  if (!mv_aligned16(a->x) || !mv_aligned16(a->w) || !mv_aligned16(a->out) || a->x_stride % vec || a->out_stride % vec) return MV_E_ALIGN;
  MoeLinear p{a->x, a->w, a->out, a->tokens, a->tiles, a->in_scale, a->x_stride, a->out_stride, (int64_t)a->n * a->k * (a->act ? 2 : 1), a->n, a->k, {}};
  if (a->act) {
    if (int e = mv_check_act(a->act)) return e;
    p.act = *a->act;
  }
  hipStream_t st = (hipStream_t)stream;
  if (dtype == MV_F32) {
    if (a->tile_m != 16) return MV_E_SHAPE;
    const dim3 grid((a->n + 63) / 64, a->max_tiles);
    if (a->act) hipLaunchKernelGGL((moe_f32_kernel<true>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((moe_f32_kernel<false>), grid, dim3(256), 0, st, p);
    MV_LAUNCH_CHECK();
    return MV_OK;
  }
  if (dtype == MV_BF16) return a->act ? launch_linear<bf16_tag, true>(p, a->tile_m, a->max_tiles, st) : launch_linear<bf16_tag, false>(p, a->tile_m, a->max_tiles, st);
  return a->act ? launch_linear<f16_tag, true>(p, a->tile_m, a->max_tiles, st) : launch_linear<f16_tag, false>(p, a->tile_m, a->max_tiles, st);
}

namespace {
// scratch memory of mv_moe_mlp: where its parts begin, in bytes
struct MlpParts {
  int64_t tokens, tiles, weights, z, end, max_tiles;
};
MlpParts mlp_parts(int rows, int top, int experts, int tile_m, int ff, int dtype) {
  const auto up = [](int64_t v) { return (v + 255) & ~(int64_t)255; };
  const int64_t pairs = (int64_t)rows * top, each = up(pairs * 4);
  MlpParts m;
  m.max_tiles = pairs / (tile_m & 0xffff) + experts;
  m.tokens = each, m.tiles = 2 * each, m.weights = m.tiles + up(m.max_tiles * 12), m.z = m.weights + each;
  m.end = m.z + pairs * ff * (dtype == MV_F32 ? 4 : 2);
  return m;
}
}  // namespace

extern "C" size_t mv_moe_mlp_workspace_bytes(int rows, int top, int experts, int tile_m, int ff, int dtype) {
  if (rows <= 0 || top <= 0 || experts <= 0 || (tile_m & 0xffff) <= 0 || ff <= 0) return 0;
  return (size_t)mlp_parts(rows, top, experts, tile_m, ff, dtype).end;
}

extern "C" int mv_moe_mlp(const MvMoeMlpArgs *a, int dtype, void *stream) {
  if (!a) return MV_E_NULLPTR;
  if (a->rows == 0) return MV_OK;
  if (!a->workspace || !a->weights || !a->place || !a->out || !a->act) return MV_E_NULLPTR;
  if (dtype != MV_BF16 && dtype != MV_F16 && dtype != MV_F32) return MV_E_DTYPE;
  if (a->rows < 0 || a->top <= 0 || (int64_t)a->rows * a->top > INT32_MAX || a->experts <= 0 || (a->tile_m & 0xffff) <= 0 || a->ff <= 0 ||
      a->router_k > a->k || a->outputs < a->experts)
    return MV_E_SHAPE;
  const MlpParts m = mlp_parts(a->rows, a->top, a->experts, a->tile_m, a->ff, dtype);
  if (!mv_aligned16(a->workspace)) return MV_E_ALIGN;
  if (a->ws_bytes < m.end || m.max_tiles > INT32_MAX) return MV_E_SHAPE;
  char *ws = (char *)a->workspace;
  int32_t *ids = (int32_t *)ws, *tokens = (int32_t *)(ws + m.tokens), *tiles = (int32_t *)(ws + m.tiles);
  float *by_place = a->weigh_inputs ? (float *)(ws + m.weights) : nullptr;
  const int pairs = a->rows * a->top, max_tiles = (int)m.max_tiles;
  // (few tokens are grouped by the router's workgroup)
  const RouteGroups few{a->place, tokens, tiles, by_place, a->experts, a->tile_m & 0xffff, max_tiles};
  bool grouped = false;
  if (int rc = route(a->x, a->x_stride, a->router, a->correction, ids, a->weights, a->rows, a->router_k, a->outputs, a->top, a->groups, a->keep, a->scale,
                     a->route_flags, dtype, stream, &few, &grouped))
    return rc;
  if (!grouped)
    if (int rc = mv_moe_group(ids, pairs, a->top, a->experts, a->tile_m & 0xffff, max_tiles, a->place, tokens, tiles, by_place ? a->weights : nullptr, by_place, stream))
      return rc;
  MvMoeLinearArgs p{};
  p.x = a->x, p.w = a->gate_up, p.out = ws + m.z, p.tokens = tokens, p.tiles = tiles, p.act = a->act, p.in_scale = by_place;
  p.x_stride = a->x_stride, p.out_stride = a->ff, p.max_tiles = max_tiles, p.tile_m = a->tile_m, p.n = a->ff, p.k = a->k;
  if (int rc = mv_moe_linear(&p, dtype, stream)) return rc;
  p.x = ws + m.z, p.w = a->down, p.out = a->out, p.tokens = nullptr, p.act = nullptr, p.in_scale = nullptr;
  p.x_stride = a->ff, p.out_stride = a->width, p.n = a->width, p.k = a->ff;
  return mv_moe_linear(&p, dtype, stream);
}
