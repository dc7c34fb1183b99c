// fp32 numbers as sums of three of bf16 (K2 and K21 in fp32).
#pragma once
#include "latent.h"

// Eight numbers as three times eight of bf16 whose sums they are (24 bits of significand, of which each part takes eight): a part is what rounding has left of the
// parts before.  ANY: also numbers that bf16 rounds to infinity, whose first part is cut off instead, and those that are not finite, which have no second
// and third part; without it all of these have a third part that is NaN.
template <bool ANY>
__device__ __forceinline__ void split3(float (&f)[8], u32x4 (&part)[3]) {
#pragma unroll
  for (int s = 0; s < 3; ++s)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t v = pack_pair<bf16_tag>(f[2 * i], f[2 * i + 1]);
      if (s < 2) {
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
      }
      part[s][i] = v;
    }
}
