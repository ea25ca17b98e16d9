// Products of more than 64 rows: y = x W^T, and gated units of it, on the tiles of the
// routed experts' products (moe_tiles_kernel.h).  Where tiles are fewer than CUs, blocks
// have shares of the contraction, whose sums in 32 bits a second kernel adds.
#include "linear_tiles.h"
#include "moe_tiles_kernel.h"

// Where these products run, and how.  Time is taken to be that of the rounds that blocks
// make, a stage of 64 columns 1.35 us in tiles of 256 rows and .9 in tiles of 128 (fitted;
// the best tile and shares of those tried are .5% faster on average), and of the sums'
// second kernel.
//   Gated units save a pass over both halves, so they are here unless the tiles fill their
// last round badly, beside a library at .95 to 1.5 PFLOP/s by its contraction: over 12
// widths, 11 contractions of 512 to 8192 and 65 to 8192 rows 1.32 times faster on average
// where chosen (from 2.0 at 512 columns to 1.04 at 8192), 1 of 1409 sizes slower by 3% (us,
// there and here: 1905 rows of 4096 into 2 x 14336 385, 361; 6000 of 3584 1083, 928; 1000
// of 2048 into 2 x 8192 65, 53; 8192 of 2048 467, 411; but 600 of 4096 140, 160).
//   Long contractions into few columns leave the library with few tiles: it takes those of
// 256 x 256, one after the other over the contraction, so the rule counts them.  Library's
// time over that here, 65 to 8192 rows, 12 widths from 1024, 11 contractions: chosen ones
// 1.48 times on average, 55 of 1983 slower (by 3 to 16%); above 16384 columns 1.98 (9 of
// 789), 13824 to 16384 1.26 (21 of 697), 11008 and 12288 1.18 (14 of 371).  With 81 to 128
// tiles, 11008 and 12288: 1.09 (16 of 78), 13824 and 14336: 1.17 (6 of 86), above 16384
// 1.49 (9 of 147).  With 129 to 256 the library's kernel may be a good one or take twice as
// long (14336 into 3584: 3684 rows 466 and 272, 4096 rows 273 and 299; 1.03, 271 of 390).
// From 8192 on only into a fifth as many columns: 1.07 (11 of 126; 65 rows of 8192 into
// 1024 1.23), above 40 tiles .94.  Rows of whole 32 KB meet few of the memory's channels,
// which shares in tiles of 128 rows show: 65 rows of 16384 into 8192 63 and 107.
extern "C" int linear_tiles_plan(long M, long O, long K, int act, bool bias, int* shares) {
  *shares = 1;
  if (M <= 64 || K < 192 || K % 64 || O < 64 || O % 64 || (act && bias)) return 0;
  const long across = ((M + 255) / 256) * ((O + 255) / 256);
  const bool plain = K < 10240 ? K >= 8192 && K >= 5 * O && across <= 40
                               : K >= (K % 16384 ? 2 : 3) * O && across <= (K < 13312 ? 80 : 128);
  if (!act && (!plain || O < 1024)) return 0;
  const long stages = K / 64;
  const int most = act ? 1 : 16;
  double least = 0;
  int found = 0;
  for (int tile = 128; tile <= 256; tile += 128) {
    const long tiles = ((M + tile - 1) / tile) * ((O + (act ? 127 : 255)) / (act ? 128 : 256));
    for (int s = 1; s <= most && stages / s >= 3 && (s == 1 || tiles * s <= 1024); ++s) {
      const double round = (double)((stages + s - 1) / s) * (tile == 256 ? 1.35 : 0.9) +
                           (tile == 256 ? 4 : 3);
      double t = (double)((tiles * s + 255) / 256) * round + 5;
      if (s > 1 || bias) t += 3 + (double)s * M * O * 8 / 5.2e6;
      if (found && t >= least) continue;
      least = t;
      found = tile;
      *shares = s;
    }
  }
  if (act) {
    const double rate = (K < 6144 ? 0.95 + K * 0.09 / 1024 : 1.5) * 1e9;
    const double there = 10 + 4.0 * M * O * K / rate + 6.0 * M * O / 4.9e6;
    if (least >= there) return 0;
  }
  return found;
}

// y [M, O] of parts [S, M, O], eight columns a thread; bound by memory
__global__ __launch_bounds__(256) void linear_parts_kernel(
    const float* __restrict__ parts, const __bf16* __restrict__ bias,
    __bf16* __restrict__ y, int M, int O, int S) {
  const long n8 = (long)M * (O / 8);
  const long at = (long)blockIdx.x * 256 + threadIdx.x;
  if (at >= n8) return;
  float v[8] = {};
  const float* p = parts + at * 8;
#pragma unroll 4
  for (int s = 0; s < S; ++s, p += n8 * 8)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const float4v f = *reinterpret_cast<const float4v*>(p + q * 4);
#pragma unroll
      for (int r = 0; r < 4; ++r) v[q * 4 + r] += f[r];
    }
  const int col = (int)(at % (O / 8)) * 8;
  bf16x8_t out;
#pragma unroll
  for (int r = 0; r < 8; ++r) out[r] = (__bf16)(v[r] + (bias ? (float)bias[col + r] : 0.0f));
  *reinterpret_cast<bf16x8_t*>(y + at * 8) = out;
}

template <int MT>
static void linear_tiles_go(MoeTilesArgs& a, int act, hipStream_t stream) {
  if (a.parts) moe_tiles_go<MT, MT_PARTS, true>(a, stream);
  else if (act == 1) moe_tiles_go<MT, MT_SILU, true>(a, stream);
  else if (act == 2) moe_tiles_go<MT, MT_GELU, true>(a, stream);
  else moe_tiles_go<MT, MT_SUMS, true>(a, stream);
}

extern "C" void launch_linear_tiles(const LinearTilesArgs* g, int tile, hipStream_t stream) {
  MoeTilesArgs a = {};
  a.x = (const char*)g->x;
  a.w = (const char*)g->w;
  a.w2 = a.w + (long)g->O * g->ldw;
  a.y = (__bf16*)g->y;
  a.xstride = g->ldx;
  a.ldw = (unsigned)g->ldw;
  a.O = g->O;
  a.K = g->K;
  a.rows = g->M;
  a.shares = g->shares;
  a.parts = g->parts;
  if (tile == 256) linear_tiles_go<256>(a, g->act, stream);
  else linear_tiles_go<128>(a, g->act, stream);
  if (!g->parts) return;
  const long n8 = (long)g->M * (g->O / 8);
  linear_parts_kernel<<<dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, stream>>>(
      a.parts, (const __bf16*)g->bias, a.y, g->M, g->O, g->shares);
}
