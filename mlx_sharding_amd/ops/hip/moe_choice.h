// A token's experts, by a wave: softmax over up to 64 logits, a lane each, and the
// lane's place among them.
#pragma once

#include "hip_common.h"

// z: the lane's logit (-INFINITY from lane `experts` on).  A lane's place is the number
// of experts before it, by weight and then by number (as bits, so also where a row is
// not a number).  True where the lane's expert is one of the first `top`: at `place`,
// with `weight`.  The exponential is the exact one: with the fast one small weights were
// off by 1.6e-6 (4e-7 so, as in torch's softmax; 32768 tokens 22.3 us, 23.0 so).
__device__ __forceinline__ bool chosen_expert(float z, int lane, int experts, int top,
                                              bool normalize, float scaling, int& place,
                                              float& weight) {
  const float most = wave_max(z);
  const float p = lane < experts ? expf(z - most) : 0.0f;
  const float share = p / wave_sum(p);
  const int key = __float_as_int(share) & 0x7FFFFFFF;
  place = 0;
#pragma unroll
  for (int i = 0; i < 64; ++i) {
    const int k = __builtin_amdgcn_readlane(key, i);
    place += k > key || (k == key && i < lane);
  }
  const bool chosen = place < top && lane < experts;
  weight = share;
  if (normalize) weight /= wave_sum(chosen ? share : 0.0f) + 1e-20f;
  weight *= scaling;
  return chosen;
}
