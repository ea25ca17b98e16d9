// Products of many rows (linear_tiles.hip); part of both extensions.
#pragma once

#include <hip/hip_runtime.h>

// x [M, K], w [O, K] (act: [2 O, K]), rows of both at multiples of 16 bytes (ldx, ldw:
// bytes, below 2^23), y [M, O]; O and K are multiples of 64, K at least 192.  act 0: none,
// 1: silu, 2: gelu_tanh.  parts [shares, M, O]: where there is a bias (per row of w) or
// more than one share, without a unit.
struct LinearTilesArgs {
  const void *x, *w, *bias;
  void* y;
  float* parts;
  int M, O, K, act, shares;
  long ldx, ldw;
};

extern "C" {
// The tile (0: the library has it) and the shares of a product.
int linear_tiles_plan(long M, long O, long K, int act, bool bias, int* shares);
void launch_linear_tiles(const LinearTilesArgs*, int tile, hipStream_t);
}
