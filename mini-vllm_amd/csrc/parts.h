// fp32 numbers as sums of three of bf16 (K2 and K21 in fp32).
#pragma once
#include "latent.h"

// Eight numbers as three times eight of bf16 whose sums they are (24 bits of significand, of which each part takes eight): a part is what rounding has left of the
// parts before.  ANY: also numbers that bf16 rounds to infinity, whose first part is cut off instead; those that are not finite, which have no second
// and third part; and those below 2^-109 some of whose bits are below 2^-133, the smallest of bf16: their own 32 bits are the first and second part, and the
// third is NaN, so that no product with them passes for a number (joined8 gives them back).  Without ANY what bf16 rounds to infinity and what is not
// finite has a third part that is NaN, and small numbers lose those bits.
template <bool ANY>
__device__ __forceinline__ void split3(float (&f)[8], u32x4 (&part)[3]) {
  uint32_t lost = 0;
#pragma unroll
  for (int s = 0; s < 3; ++s)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t v = pack_pair<bf16_tag>(f[2 * i], f[2 * i + 1]);
      if (ANY || s < 2) {
        const float lo = u2f(v << 16), hi = u2f(v & 0xffff0000u);
        float rl = f[2 * i] - lo, rh = f[2 * i + 1] - hi;
        if (ANY && s == 0 && (!(fabsf(lo) < INFINITY) || !(fabsf(hi) < INFINITY))) {
          auto cut = [](float x, float first, float &rest) {
            if (fabsf(first) < INFINITY) return f2u(first);
            const uint32_t top = f2u(x) & 0xffff0000u;
            if (fabsf(x) < INFINITY) {
              rest = x - u2f(top);
              return top;
            }
            rest = 0.f;
            return x != x ? top | 0x400000u : top;
          };
          const uint32_t a = cut(f[2 * i], lo, rl), b = cut(f[2 * i + 1], hi, rh);
          v = a >> 16 | b;
        }
        f[2 * i] = rl, f[2 * i + 1] = rh;
        if (ANY && s == 2) lost |= f2u(rl) | f2u(rh);
      }
      part[s][i] = v;
    }
  if (ANY && lost & 0x7fffffffu) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if ((f2u(f[i]) & 0x7fffffffu) == 0) continue;
      const int shift = i & 1 ? 16 : 0;
      auto of = [&](int s) { return u2f(i & 1 ? part[s][i >> 1] & 0xffff0000u : part[s][i >> 1] << 16); };
      const uint32_t own = f2u(of(0) + (of(1) + (of(2) + f[i]))), to[3] = {own >> 16, own & 0xffffu, 0x7fc0u};   // (exact sums)
#pragma unroll
      for (int s = 0; s < 3; ++s) part[s][i >> 1] = part[s][i >> 1] & (0xffff0000u >> shift) | to[s] << shift;
    }
  }
}

// The numbers whose parts these are
__device__ __forceinline__ void joined8(const u32x4 (&part)[3], float (&f)[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    auto of = [&](int s) { return i & 1 ? part[s][i >> 1] & 0xffff0000u : part[s][i >> 1] << 16; };
    const float third = u2f(of(2));
    f[i] = third != third ? u2f(of(0) | of(1) >> 16) : u2f(of(0)) + (u2f(of(1)) + third);
  }
}
