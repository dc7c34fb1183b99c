// K7 (+ per-head K6, + K1) — q/k head RMSNorm -> rotary embedding (NeoX halves or interleaved pairs) ->
// K/V cache store in ONE launch
// (reference: minivllm/models/qwen_base.py:173-190 flat path,
//  layers/layernorm.py:81-93, layers/rotary_embedding.py:77-81,166-193,
//  layers/attention_backend.py:196-266).
// One workgroup per token, of one, two or four waves.  A head row (D elements) is spread over
// LPT = D/VEC adjacent lanes, 16 bytes each; the rotation partner
// (dims i and i + D/2) lives LPT/2 lanes away and is fetched with one DPP
// row rotate (bf16/f16, D=128) or a wave shuffle.
// Rounding points are the reference's: norm result -> dtype, rotation in
// fp32 with separately rounded products -> dtype.
#include <algorithm>

#include "common.h"

struct RopeParams {
  const void *q, *k, *v;
  int64_t q_stride, k_stride, v_stride;
  const int64_t *positions;
  const float *cos, *sin;
  int64_t max_pos;
  const void *q_norm_w, *k_norm_w;
  float eps;
  int norm_dim;   // columns that the head norms are means over
  int unit;       // rows divided by their rms, no weight, one rounding behind the rotation
  void *q_out, *k_out, *k_cache, *v_cache;
  const int32_t *slot_mapping;
  int64_t num_slots;
  int n_heads, n_kv_heads;
  int pairs, interleaved;   // rotary layout (common.h: rot_factors)
};

template <int LPT>
__device__ __forceinline__ float lpt_sum(float x) {
  // butterfly over the LPT lanes of one head row; every lane gets the total
  if constexpr (LPT <= 16) return lanes_sum<LPT>(x);   // (the same sums, without the LDS pipe)
  for (int off = 1; off < LPT; off <<= 1) x += __shfl_xor(x, off, 64);
  return x;
}

// Rows of a token, 16 bytes a lane.  A thread reads its cosines and sines once, 64 bytes for 16 of each row, so that they are more of what passes through
// the L1 than the rows themselves where a thread has two or three rows: with many tokens a token is one wave (two), which asks for four of its rows at a time; with few,
// whose time is one token's latency, four waves, a row each at a time.
template <typename Tag, int D, int THREADS>
__global__ void __launch_bounds__(THREADS) rope_qk_store_kernel(RopeParams p) {
  typedef typename elem<Tag>::T T;
  constexpr int VEC = elem<Tag>::VEC;
  constexpr int LPT = D / VEC;
  const int tok = blockIdx.x;
  const int sub = threadIdx.x % LPT;
  constexpr int rows_per_iter = THREADS / LPT;
  const int H = p.n_heads, HKV = p.n_kv_heads;
  const bool has_cache = p.k_cache != nullptr && p.slot_mapping != nullptr;
  int64_t slot = has_cache ? (int64_t)p.slot_mapping[tok] : -1;
  if (slot >= p.num_slots) slot = -1;
  const int total_rows = H + HKV + (has_cache ? HKV : 0);
  const int64_t pos = p.positions[tok];
  constexpr int AHEAD = THREADS < 256 ? 4 : 1;
  const auto source = [&](int r) {
    return r < H          ? (const T *)p.q + (int64_t)tok * p.q_stride + r * D
           : r < H + HKV ? (const T *)p.k + (int64_t)tok * p.k_stride + (r - H) * D
                         : (const T *)p.v + (int64_t)tok * p.v_stride + (r - H - HKV) * D;
  };
  const int first = threadIdx.x / LPT;
  u32x4 raws[AHEAD];
  const auto ask = [&](int r0) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) raws[u] = *reinterpret_cast<const u32x4 *>(source(min(r0 + u * rows_per_iter, total_rows - 1)) + sub * VEC);
  };
  ask(first);
  const bool pos_ok = pos >= 0 && pos < p.max_pos;
  float cs[VEC], sn[VEC];
  rot_factors<D, VEC>(p.cos, p.sin, pos, pos_ok, sub, p.pairs, p.interleaved != 0, cs, sn);

  for (int r0 = first; r0 - first < total_rows; r0 += AHEAD * rows_per_iter) {
    if (r0 != first) ask(r0);
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const int r = r0 + u * rows_per_iter;
      if (r >= total_rows) continue;   // (the lanes of a row together)
      if (r >= H + HKV) {  // raw V row -> cache
        if (slot >= 0) *reinterpret_cast<u32x4 *>((T *)p.v_cache + (slot * HKV + r - H - HKV) * D + sub * VEC) = raws[u];
        continue;
      }
      const bool is_q = r < H;
      const int hh = is_q ? r : r - H;
      const T *nw = is_q ? (const T *)p.q_norm_w : (const T *)p.k_norm_w;
      float x[VEC];
      if constexpr (VEC == 8) unpack8<Tag>(raws[u], x);
      else {
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = u2f(raws[u][j]);
      }
      float rs = 1.0f;
      if (nw != nullptr || p.unit) {   // (a rotation keeps the length)
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < VEC; ++j) ss = fmaf(x[j], x[j], ss);
        ss = lpt_sum<LPT>(ss);
        rs = 1.0f / sqrtf(ss / (float)p.norm_dim + p.eps);
      }
      if (nw != nullptr) {  // per-head RMSNorm, result rounded to dtype like the reference
        float w[VEC];
        const u32x4 wraw = *reinterpret_cast<const u32x4 *>(nw + sub * VEC);
        if constexpr (VEC == 8) unpack8<Tag>(wraw, w);
        else {
#pragma unroll
          for (int j = 0; j < 4; ++j) w[j] = u2f(wraw[j]);
        }
#pragma unroll
        for (int j = 0; j < VEC; ++j)
          x[j] = elem<Tag>::ld(elem<Tag>::st(__fmul_rn(__fmul_rn(x[j], rs), w[j])));
      }
      float y[VEC];
      rot_apply<D, VEC>(x, cs, sn, sub, p.interleaved != 0, y);
      if (p.unit) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) y[j] = __fmul_rn(y[j], rs);
      }
      u32x4 packed;
      if constexpr (VEC == 8) packed = pack8<Tag>(y);
      else {
#pragma unroll
        for (int j = 0; j < 4; ++j) packed[j] = f2u(y[j]);
      }
      if (is_q) {
        *reinterpret_cast<u32x4 *>((T *)p.q_out + ((int64_t)tok * H + hh) * D + sub * VEC) = packed;
      } else {
        if (p.k_out != nullptr) *reinterpret_cast<u32x4 *>((T *)p.k_out + ((int64_t)tok * HKV + hh) * D + sub * VEC) = packed;
        if (slot >= 0) *reinterpret_cast<u32x4 *>((T *)p.k_cache + (slot * HKV + hh) * D + sub * VEC) = packed;
      }
    }
  }
}

// Waves of a token.  A wave has its rows one batch of four behind the other, a norm about doubles what a batch takes, and tokens beside each other on a SIMD cover that:
// the more rows, the more tokens it takes until fewer waves are ahead; up to 768 tokens there are at most three workgroups to a CU, of four waves or of two.  bf16, us by 4 / 2 / 1
// waves, launches of a graph.  With norms: 16 + 8 heads of 128 (rows of q, k and v: 32) 513 tokens 6.5 / 6.1 / 7.2, 780 8.3 / 7.3 / 7.7, 1200 10.0 / 8.9 / 9.4, 1600 12.7 / 10.9 /
// 10.4; 24 + 8 513 6.9 / 7.3 / 8.6; 40 + 8 (56 rows) 720 9.1 / 9.7 / 11.6, 780 10.5 / 9.9 / 11.8, 1024 11.3 / 10.6 / 12.6, 1450 14.8 / 15.5 / 16.1; 64 + 8 (80) 720 11.2 / 12.5 / 15.5, 900
// 13.9 / 14.1 / 16.7, 1450 17.8 / 19.9 / 21.2, 2800 28.5 / 27.9 / 29.0; 16 + 4 of 256 (24) 513 10.8 / 10.3 / 13.3, 1450 19.5 / 17.4 / 17.6, 1900 23.5 / 20.2 / 19.4; 32 + 8 of 256 (48) 1100
// 22.7 / 23.3 / 29.2, 1900 30.1 / 28.3 / 30.9, 3500 48.0 / 45.5 / 42.0.  Without: 28 + 4 of 128 (36) 513 6.0 / 5.8 / 6.6, 1024 8.2 / 7.4 / 7.4; 64 + 8 720 .. 760 9.3 / 9.4 / 11.7, 780 10.5 / 9.8 /
// 11.9, 1450 15.8 / 14.8 / 14.8, 1900 18.9 / 17.8 / 16.6; 40 + 40 of 128 (120) 520 11.2 / 11.7 / 15.8, 2800 37.6 / 35.4 / 35.2, 8000 112.8 / 118.3 / 122.6; more than six batches of a
// single wave: 32 + 16 of 256 with norms 4000 72.6 / 72.6 / 76.5.  Over 23 shapes of 18 to 96 rows, 513 to 5000 tokens (269 pairs): 0.93 of four waves' time in the mean, at worst
// 6 % above the best.  fp32 rows are as quick either way (16 + 8 of 128, 5000: 33.8 / 34.4 / 33.1) and slower below (1000: 10.7 / 11.7 / 16.2).
static int waves_of_token(const RopeParams &p, int head_dim, int n_tok) {
  const int rows = p.n_heads + (p.k_cache ? 2 : 1) * p.n_kv_heads, wide = head_dim == 256 ? rows * 3 / 2 : rows;
  const bool norm = p.q_norm_w || p.unit;
  if (rows > 100 || n_tok <= 512) return 4;
  if (n_tok > (norm ? 44 * wide : std::min(25 * wide, 1400)) && rows * head_dim <= 6 * 4 * 512) return 1;
  return n_tok > (norm && rows > 64 ? 2048 : rows > (norm ? 36 : 64) ? 768 : 512) ? 2 : 4;
}

template <typename Tag, int D>
static void launch_rope(const RopeParams &p, int n_tok, hipStream_t st) {
  const int waves = elem<Tag>::VEC == 8 ? waves_of_token(p, D, n_tok) : 4;
  if constexpr (elem<Tag>::VEC == 8) {
    if (waves == 1) hipLaunchKernelGGL((rope_qk_store_kernel<Tag, D, 64>), dim3(n_tok), dim3(64), 0, st, p);
    if (waves == 2) hipLaunchKernelGGL((rope_qk_store_kernel<Tag, D, 128>), dim3(n_tok), dim3(128), 0, st, p);
  }
  if (waves == 4) hipLaunchKernelGGL((rope_qk_store_kernel<Tag, D, 256>), dim3(n_tok), dim3(256), 0, st, p);
}

extern "C" int mv_rope_qk_store_ex(const void *q, const void *k, const void *v, int64_t q_stride_tok,
                                int64_t k_stride_tok, int64_t v_stride_tok,
                                const int64_t *positions, const float *cos, const float *sin,
                                int64_t max_pos, const void *q_norm_w, const void *k_norm_w,
                                float eps, void *q_out, void *k_out, void *k_cache, void *v_cache,
                                const int32_t *slot_mapping, int64_t num_slots, int n_tok,
                                int n_heads, int n_kv_heads, int head_dim, int dtype,
                                const MvAttnOpts *opts, void *stream) {
  if (n_tok == 0) return MV_OK;
  if (!q || !k || !positions || (mv_needs_tables(opts) && (!cos || !sin)) || !q_out) return MV_E_NULLPTR;
  if ((q_norm_w == nullptr) != (k_norm_w == nullptr)) return MV_E_NULLPTR;
  if (q_norm_w && opts && opts->unit_norm) return MV_E_SHAPE;
  const bool has_cache = k_cache != nullptr || v_cache != nullptr || slot_mapping != nullptr;
  if (has_cache && (!k_cache || !v_cache || !slot_mapping || !v)) return MV_E_NULLPTR;
  if (n_tok < 0 || n_heads <= 0 || n_kv_heads <= 0 || (mv_needs_tables(opts) && max_pos <= 0)) return MV_E_SHAPE;
  if (head_dim != 64 && head_dim != 128 && head_dim != 256) return MV_E_SHAPE;
  if (int e = mv_check_rot(opts, head_dim)) return e;
  if (dtype != MV_BF16 && dtype != MV_F16 && dtype != MV_F32) return MV_E_DTYPE;
  const int esz = dtype == MV_F32 ? 4 : 2;
  if (!mv_aligned16(q) || !mv_aligned16(k) || !mv_aligned16(q_out) ||
      (v && !mv_aligned16(v)) || (k_out && !mv_aligned16(k_out)) ||
      (k_cache && !mv_aligned16(k_cache)) || (v_cache && !mv_aligned16(v_cache)) ||
      (q_norm_w && (!mv_aligned16(q_norm_w) || !mv_aligned16(k_norm_w))) ||
      (q_stride_tok * esz) % 16 || (k_stride_tok * esz) % 16 || (v_stride_tok * esz) % 16)
    return MV_E_ALIGN;
  RopeParams p;
  p.q = q; p.k = k; p.v = v;
  p.q_stride = q_stride_tok; p.k_stride = k_stride_tok; p.v_stride = v_stride_tok;
  p.positions = positions; p.cos = cos; p.sin = sin; p.max_pos = max_pos;
  p.q_norm_w = q_norm_w; p.k_norm_w = k_norm_w; p.eps = eps;
  p.q_out = q_out; p.k_out = k_out;
  p.k_cache = has_cache ? k_cache : nullptr;
  p.v_cache = has_cache ? v_cache : nullptr;
  p.slot_mapping = has_cache ? slot_mapping : nullptr;
  p.num_slots = num_slots;
  p.n_heads = n_heads; p.n_kv_heads = n_kv_heads;
  p.norm_dim = opts && opts->norm_dim ? opts->norm_dim : head_dim;
  p.unit = opts && opts->unit_norm;
  p.interleaved = opts && opts->interleaved;
  p.pairs = p.interleaved ? opts->rot_pairs : head_dim / 2;
  hipStream_t st = (hipStream_t)stream;
  if (head_dim == 256) {
    MV_DISPATCH_DTYPE(dtype, (launch_rope<Tag, 256>(p, n_tok, st)));
  } else if (head_dim == 128) {
    MV_DISPATCH_DTYPE(dtype, (launch_rope<Tag, 128>(p, n_tok, st)));
  } else {
    MV_DISPATCH_DTYPE(dtype, (launch_rope<Tag, 64>(p, n_tok, st)));
  }
  MV_LAUNCH_CHECK();
  return MV_OK;
}

extern "C" int mv_rope_qk_store(const void *q, const void *k, const void *v, int64_t q_stride_tok,
                                int64_t k_stride_tok, int64_t v_stride_tok,
                                const int64_t *positions, const float *cos, const float *sin,
                                int64_t max_pos, const void *q_norm_w, const void *k_norm_w,
                                float eps, void *q_out, void *k_out, void *k_cache, void *v_cache,
                                const int32_t *slot_mapping, int64_t num_slots, int n_tok,
                                int n_heads, int n_kv_heads, int head_dim, int dtype,
                                void *stream) {
  return mv_rope_qk_store_ex(q, k, v, q_stride_tok, k_stride_tok, v_stride_tok, positions, cos, sin, max_pos, q_norm_w,
                             k_norm_w, eps, q_out, k_out, k_cache, v_cache, slot_mapping, num_slots, n_tok, n_heads,
                             n_kv_heads, head_dim, dtype, nullptr, stream);
}
