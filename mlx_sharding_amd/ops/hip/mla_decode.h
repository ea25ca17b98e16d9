// Arguments of latent attention of one token per sequence (mla_decode.hip).
#pragma once

#include "hip_common.h"

// nope and rank are multiples of 32, rope is even, q rows begin at 16 bytes
struct MlaPrepareArgs {
  const __bf16 *q, *latent;   // [N, heads * (nope + rope)], [N, rank + rope]
  const __bf16 *w, *norm;     // [heads, rank, nope], [rank]
  const float *cos, *sin;     // [rope / 2] of the token's position
  __bf16 *out, *cache;        // [N, heads, rank + rope], [N, cap, rank + rope]
  const int* pos;             // the row's place, or null: pos0
  long ld_q, ld_latent, cap, pos0;
  int N, heads, nope, rope, rank;
  float eps, offset;
};

// up to 64 slices of whole tiles of keys; rank a multiple of 32, vdim of 16
struct MlaFinishArgs {
  const float *part_o, *part_ml;  // of attn_decode.hip, rank columns
  const __bf16* w;                // [heads, vdim, rank]
  __bf16* out;                    // [N, heads, vdim]
  const int* pos;                 // of the last key, or null: `keys` of them
  int N, heads, rank, vdim, slices, tile, keys;
};

// Rows of a prompt.  rank and rope are multiples of 8, all rows begin at 16 bytes.
struct MlaRowsArgs {
  const __bf16 *latent, *norm;  // [B * T, rank + rope], [rank]
  const float *cos, *sin;       // [T, rope / 2]
  __bf16 *cache, *rows;         // [B, cap, rank + rope], [B * T, rank] or null
  long ld_latent, cap, pos0, N;
  int T, rank, rope;
  float eps, offset;
};

extern "C" {
void launch_mla_rows(const MlaRowsArgs*, hipStream_t);
void launch_mla_prepare(const MlaPrepareArgs*, hipStream_t);
void launch_mla_finish(const MlaFinishArgs*, hipStream_t);
}
