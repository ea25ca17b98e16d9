// Routed experts of a prompt: choice of the experts, places of the (token, expert)
// pairs, sorted by expert and cut into tiles of one expert, and the two matrix products
// over the tiles (moe_tiles_kernel.h).
// Measured: 32768 tokens, top 6 of 64 experts of 2048 x 1408, the layer 4.39 -> 3.34 ms;
// 4096 tokens 851 -> 546 us, 200 tokens 458 -> 246 (the weights alone take 225).  Before:
// pairs scattered to experts padded to the fullest one (its count read back by the
// host), two batched library products on transposed copies of the weights, the unit in
// between.

#include "moe_tiles_kernel.h"
#include "moe_choice.h"

// ---------------------------------------------------------------------------
// Experts of the tokens, a wave each.  Bound by its instructions, five for each pair of
// experts.  For 32768 tokens of 64 experts softmax, selection, sorting, scaling and
// conversions of their own took 160 us (the selection alone 119); 23 here.
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void moe_choose_kernel(
    const __bf16* __restrict__ logits, long* __restrict__ choice,
    float* __restrict__ weight, int N, int E, int top, int normalize, float scaling) {
  const int lane = threadIdx.x & (WAVE - 1);
  const long t = (long)blockIdx.x * 4 + threadIdx.x / WAVE;
  if (t >= N) return;
  int place;
  float w;
  if (chosen_expert(lane < E ? (float)logits[t * E + lane] : -INFINITY, lane, E, top,
                    normalize, scaling, place, w)) {
    choice[t * top + place] = lane;
    weight[t * top + place] = w;
  }
}

// logits bf16 [N, E], E up to 64, top up to E
extern "C" void launch_moe_choose(const void* logits, long* choice, float* weight, int N,
                                  int E, int top, int normalize, float scaling,
                                  hipStream_t stream) {
  moe_choose_kernel<<<dim3((unsigned)((N + 3) / 4)), dim3(256), 0, stream>>>(
      (const __bf16*)logits, choice, weight, N, E, top, normalize, scaling);
}

// ---------------------------------------------------------------------------
// Places.  Pairs of an expert lie in any order within those of a block: a pair's
// result does not depend on its place.
// ---------------------------------------------------------------------------

__device__ __forceinline__ int pair_expert(const MoePlaceArgs& a, int p) {
  return (int)min(max(a.choice[p], 0L), (long)a.experts - 1);
}

__global__ __launch_bounds__(256) void moe_count_kernel(const MoePlaceArgs a) {
  __shared__ int count[MT_EXPERTS];
  for (int e = threadIdx.x; e < a.experts; e += 256) count[e] = 0;
  __syncthreads();
  const int p0 = blockIdx.x * MT_BLOCK_PAIRS;
  for (int i = threadIdx.x; i < MT_BLOCK_PAIRS && p0 + i < a.pairs; i += 256)
    atomicAdd(&count[pair_expert(a, p0 + i)], 1);
  __syncthreads();
  for (int e = threadIdx.x; e < a.experts; e += 256)
    a.hist[(long)blockIdx.x * a.experts + e] = count[e];
}

// one block, a thread per expert
__global__ __launch_bounds__(MT_EXPERTS) void moe_plan_kernel(const MoePlaceArgs a) {
  __shared__ int pairs[MT_EXPERTS], tiles[MT_EXPERTS];
  const int e = threadIdx.x;
  int n = 0;
  if (e < a.experts) {
#pragma unroll 8
    for (int b = 0; b < a.blocks; ++b) n += a.hist[(long)b * a.experts + e];
  }
  const int nt = (n + a.tile - 1) / a.tile;
  pairs[e] = n;
  tiles[e] = nt;
  __syncthreads();
  for (int d = 1; d < MT_EXPERTS; d *= 2) {  // sums up to and with each expert
    const int x = e >= d ? pairs[e - d] : 0, y = e >= d ? tiles[e - d] : 0;
    __syncthreads();
    pairs[e] += x;
    tiles[e] += y;
    __syncthreads();
  }
  if (e == MT_EXPERTS - 1) *a.n_tiles = tiles[e];
  if (e >= a.experts) return;
  int at = pairs[e] - n;
  int* t = a.tiles + (tiles[e] - nt) * 3;
  for (int i = 0; i < nt; ++i, t += 3) {
    t[0] = e;
    t[1] = at + i * a.tile;
    t[2] = min(a.tile, n - i * a.tile);
  }
#pragma unroll 8
  for (int b = 0; b < a.blocks; ++b) {
    int* h = a.hist + (long)b * a.experts + e;
    const int c = *h;
    *h = at;
    at += c;
  }
}

__global__ __launch_bounds__(256) void moe_place_kernel(const MoePlaceArgs a) {
  __shared__ int next[MT_EXPERTS];
  for (int e = threadIdx.x; e < a.experts; e += 256)
    next[e] = a.hist[(long)blockIdx.x * a.experts + e];
  __syncthreads();
  const int p0 = blockIdx.x * MT_BLOCK_PAIRS;
  for (int i = threadIdx.x; i < MT_BLOCK_PAIRS && p0 + i < a.pairs; i += 256) {
    const int at = atomicAdd(&next[pair_expert(a, p0 + i)], 1);
    a.where[p0 + i] = at;
    a.tokens[at] = (p0 + i) / a.top;
  }
}

extern "C" void launch_moe_place(const MoePlaceArgs* a, hipStream_t stream) {
  const dim3 grid((unsigned)a->blocks), block(256);
  moe_count_kernel<<<grid, block, 0, stream>>>(*a);
  moe_plan_kernel<<<dim3(1), dim3(MT_EXPERTS), 0, stream>>>(*a);
  moe_place_kernel<<<grid, block, 0, stream>>>(*a);
}

extern "C" void launch_moe_tiles(MoeTilesArgs* a, int tile, bool gated,
                                 hipStream_t stream) {
  if (tile == 256) {
    if (gated) moe_tiles_go<256, MT_SILU>(*a, stream);
    else moe_tiles_go<256, MT_SUMS>(*a, stream);
  } else {
    if (gated) moe_tiles_go<128, MT_SILU>(*a, stream);
    else moe_tiles_go<128, MT_SUMS>(*a, stream);
  }
}
