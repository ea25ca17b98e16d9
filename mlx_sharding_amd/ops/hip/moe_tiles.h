// Arguments of the routed experts' kernels of a prompt.
#pragma once

#include "hip_common.h"

#define MT_BLOCK_PAIRS 2048  // (token, expert) pairs of a placing block
#define MT_EXPERTS 1024

struct MoePlaceArgs {
  const long* choice;  // [pairs] expert
  int* hist;           // [blocks, experts]; from moe_plan on the first place of each
  int* tiles;          // [count, 3]: expert, first pair, pairs
  int* n_tiles;
  int *where, *tokens;  // [pairs]: place of a pair, token of a place
  int pairs, top, experts, blocks, tile;
};

// What is made of the sums: themselves, silu(those with w) * those with w2 (or gelu), or
// g sigmoid(alpha g) (u + 1) of both times scale[p], g at most `limit`, u within +-limit;
// or themselves in 32 bits.
enum MoeUnit { MT_SUMS = 0, MT_SILU = 1, MT_CLAMPED = 2, MT_GELU = 3, MT_PARTS = 4 };

// y[p, o] of x[token of p] . w[expert of p, o] (and w2).  K and O are multiples of 64, K
// at least 128; rows of w begin at 16 bytes; offsets within x (tokens given) and within
// an expert's matrix below 2^32.
struct MoeTilesArgs {
  const char *x, *w, *w2;  // [rows, K], [experts, O, K]; w2: up's
  __bf16* y;               // [pairs, O]
  const int* tokens;       // of a unit: row of x of a pair; else the pair is
  const int *tiles, *n_tiles;
  long xstride;            // bytes
  int O, K, cols;          // cols: blocks across O
  long wstride;            // bytes from one expert's matrix to the next
  const float* scale;      // clamped: [pairs]
  float limit, alpha;
  unsigned ldw;            // bytes from one row of w to the next
  // dense: rows of x; parts of the contraction, and their sums [shares, rows, O]
  int rows, shares;
  float* parts;
};

extern "C" {
void launch_moe_choose(const void*, long*, float*, int, int, int, int, float, hipStream_t);
void launch_moe_place(const MoePlaceArgs*, hipStream_t);
// pairs of a tile: 256 or 128; gated: silu (moe_tiles.hip) or clamped units
// (ragged_experts_tiles.hip), else sums
void launch_moe_tiles(MoeTilesArgs*, int tile, bool gated, hipStream_t);
void launch_clamped_tiles(MoeTilesArgs*, int tile, bool gated, hipStream_t);
}
