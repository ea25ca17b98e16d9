// Arguments of the routed experts' kernels of a decoding step (moe_rows.hip).
#pragma once

#include "hip_common.h"

#define MR_PAIRS 1024  // (token, expert) pairs of a batch

struct MoeRowsArgs {
  const void* x;             // bf16 rows [N, K] (up), h rows [pairs, K] (down)
  const void *w, *w2;        // packed (moe_pack) or bf16 [E, O, K]; up: gate's, up's
  void* y;                   // up: h [pairs, O]; down: fp32 [pairs, O]
  const int* choice;         // [pairs] expert
  const float* weight;       // [pairs]
  int pairs, top, experts, O, K;
  // the token's shared feed-forward in the same launch: its first `dense` = DO / 16
  // blocks (or none).  dw: bf16 [2 DO, DK] (up: the gate's rows, the up projection's) or
  // [DO, DK] (down); rows dx [N, DK] of it, results dy [N, DO]
  const __bf16 *dx, *dw;
  __bf16* dy;
  int dense, N, DO, DK;
  unsigned by_blocks, by_rows;  // reciprocals that launch_moe_rows fills in
};
static_assert(sizeof(MoeRowsArgs) <= 128, "two lines");

struct MoeRouteArgs {
  const __bf16 *x, *residual, *norm, *gate;  // rows [N, H], [H], [E, H]
  __bf16 *h, *y;       // x + residual (if given), normed rows
  int* choice;
  float* weight;
  int H, E, top;
  float eps, offset, scaling;
  int normalize;
  float* logits;       // [N, 64], and a number per token that is 0 before: with these a
  unsigned* tickets;   // token has a block for every 16 experts
};

extern "C" {
// words of a packed tile of 16 rows by 128 of the contraction
inline int moe_pack_words(int bits, int gs) {
  return 16 * 128 * bits / 32 + 16 * (128 / gs);
}
void launch_moe_pack(const void*, const void*, const void*, void*, int, int, int,
                     int, hipStream_t);
void launch_moe_rows(const MoeRowsArgs*, int, int, bool, hipStream_t);
int moe_rows_longest(int);
// moe_shared.hip
void launch_moe_begin(const MoeRouteArgs*, int, const void*, void*, int, hipStream_t);
void launch_moe_finish(const void*, const void*, const float*, const void*, void*, int, int,
                       int, int, hipStream_t);
void launch_moe_route(const MoeRouteArgs*, int, hipStream_t);
void launch_moe_combine(const float*, const void*, const void*, void*, int, int,
                        int, hipStream_t);
}
