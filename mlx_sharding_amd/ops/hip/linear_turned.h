// Where queries, keys and values of few tokens go (linear_turned.hip).
#pragma once

#include "hip_common.h"

struct TurnedArgs {
  const float *cos, *sin;   // [T, D / 2]
  __bf16 *kcache, *vcache;  // [sequences, Hkv, cap, D], from row `at` on
  long cap, at;
  int T, Hq, Hkv;           // T: rows of a sequence
};

extern "C" {
// D: of a head, a power of two; heads: queries, keys and values
bool linear_turned_takes(long M, long heads, long D, long K);
// queries [M, Hq * D]
void launch_linear_turned(const void*, const void*, const void*, const void*, void*, int, int,
                          int, long, long, float, float, const TurnedArgs*, hipStream_t);
}
