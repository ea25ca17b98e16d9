// Capped scores, cap * tanh(s / cap), as the powers of two that softmax takes.
//
// tanh(y) = y (1 + y^2 P(y^2)) below .55, P fitted by weighted least squares to .6 of a
// unit of 32 bits; above that, 1 - 2 / (e^2y + 1), which below loses bits to its
// subtraction.  With the roundings around it either is as close as a tanh that is off by
// one unit.  Scores are rarely above: a wave that has none skips that part.  Four at a
// time, as more leave prompts of 256 columns without registers.
// Measured, a prompt of 4096 tokens, 16 heads of 256 over 8: 240 us, 228 with the
// subtraction for all scores (and errors of 2^-24 of the cap), 290 where every wave has
// scores above; decoding is bound by memory and as fast.
#pragma once

#include "hip_common.h"

struct SoftCap {
  float lin;   // score -> power of two, without the cap
  float arg;   // score -> y
  float out;   // the cap in powers of two; 0: no cap
  float p[4];  // P, times lin
};

inline SoftCap soft_cap(float scale, float cap) {
  constexpr float LOG2E = 1.44269504088896340736f;
  SoftCap c{scale * LOG2E, 0.0f, 0.0f, {}};
  if (cap > 0.0f) {
    c.arg = scale / cap;
    c.out = cap * LOG2E;
    const float p[4] = {-0.3333294689655304f, 0.13320724666118622f,
                        -5.267181247472763e-2f, 1.6437578946352005e-2f};
    for (int i = 0; i < 4; ++i) c.p[i] = p[i] * c.lin;
  }
  return c;
}

// N scores of this lane; all lanes of the wave take part
template <int N>
__device__ __forceinline__ void soft_capped(const SoftCap& c, float (&s)[N]) {
  constexpr float LIMIT = 0.55f, TWO_LOG2E = 2.88539008177792681472f;
  float most = 0.0f;
#pragma unroll
  for (int i = 0; i < N; ++i) most = fmaxf(most, fabsf(s[i]));
  auto small = [&](float x) {
    const float y = x * c.arg, z = y * y;
    float p = c.p[3];
#pragma unroll
    for (int i = 2; i >= 0; --i) p = fmaf(p, z, c.p[i]);
    return x * fmaf(p, z, c.lin);
  };
  if (!__any(most * fabsf(c.arg) >= LIMIT)) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      s[i] = small(s[i]);
      if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const float y = fabsf(s[i] * c.arg);
      const float e = __builtin_amdgcn_exp2f(y * TWO_LOG2E);
      const float t = fmaf(-2.0f * c.out, __builtin_amdgcn_rcpf(e + 1.0f), c.out);
      s[i] = y < LIMIT ? small(s[i]) : copysignf(t, s[i] * c.arg);
    }
  }
}
