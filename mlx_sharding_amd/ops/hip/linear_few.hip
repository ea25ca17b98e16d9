// y = x W^T for few rows of x (decoding, short prompts): what lies between two such products of
// a layer goes with them.
//
//   before:  RMS norm of x's rows with a weight per column
//   behind:  bias, residual rows, or the gated unit act(gate) * up of two halves
//            of W's rows
//
// Bound by reading W once; a short kernel also by launch and latency, so each
// operation taken along saves its launch (about 4 us within a captured step).
// W goes from memory to operands of 16x16x32 products (a lane: 16 bytes of one of
// 16 rows), the waves of a block take the contraction in chunks by turns and add
// up through LDS.  x comes from L2, once per block: more rows of W a block where
// there are enough of them and more than a few rows of x.  The norm's factor is
// applied to the sums: x times the weight is rounded to bf16, as the normed row
// was.
// Measured with weights out of memory (sets of 1.5 GB and more by turns), beside the
// library's product (us; M x K x O): 1 x 2048 x 2048: 5.0,
// 11.0; 1 x 4096 x 4096: 8.4, 15.5; 1 x 4096 x 28672: 38 (6.2 TB/s), 62; 16 of
// these: 48, 59; 1 x 14336 x 4096: 22.5, 26; 8 of these: 24.6, 26.6; 16: 29, 26.
// With norm and unit, 1 x 4096 x 28672: 46, beside 72 for three kernels.

#include "linear_few_kernel.h"

// RT tiles of 16 rows of W; with a gated unit half of them are the gate's, the
// others the up projection's.  SHARED: blocks have a share of a contraction each (in every
// kernel they cost 1% of the time: 9 of x, 4608 rows of 512 3.91 us so, 3.83 as it is)
template <int RT, int ACT, bool NORM, int NW, int U, bool SHARED>
__global__ __launch_bounds__(NW * WAVE) void linear_few_kernel(
    const LinearFewArgs a) {
  __shared__ __attribute__((aligned(16))) f32x4 red[NW][RT][WAVE];
  __shared__ float squares[NORM ? NW : 1][WAVE];

  arrive(a);
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int l16 = lane & 15, lg = lane >> 4;
  constexpr int YT = ACT ? RT / 2 : RT;  // tiles of y's columns
  const int row0 = blockIdx.x * 16 * YT;

  const __bf16* wp[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int row = r / YT * a.O + min(row0 + r % YT * 16 + l16, a.O - 1);
    wp[r] = a.w + (long)row * a.ldw;
  }
  const __bf16* xp = a.x + (long)min(l16, a.M - 1) * a.ldx;

  f32x4 acc[RT];
  float sq = 0.0f;
#pragma unroll
  for (int r = 0; r < RT; ++r) acc[r] = f32x4{0, 0, 0, 0};
  auto normed = [&](bf16x8_t v, bf16x8_t g) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float f = (float)v[j];
      sq = fmaf(f, f, sq);
      v[j] = (__bf16)(f * ((float)g[j] + a.offset));
    }
    return v;
  };
  auto load = [](const __bf16* p) {
    return *reinterpret_cast<const bf16x8_t*>(p);
  };

  // this block's share of the contraction
  const int s0 = SHARED ? blockIdx.y * a.share : 0;
  const int steps = SHARED ? min(a.share, a.K / 32 - s0) : a.K / 32;
  const int chunks = steps / U, first = first_of(a, a.share / U, chunks, blockIdx.x);
  // operands of one chunk; the next one's are asked for before this one is used,
  // rows of x among them, as loads come back in order
  struct Chunk {
    bf16x8_t w[RT][U], x[U], g[NORM ? U : 1];
  };
  auto fetch = [&](Chunk& f, int c) {
    c += first;
    if (c >= chunks) c -= chunks;
    // the steps of a row one after the other: two are a line of 128 bytes, of which the
    // second half is then on its way (28672 rows of 4096: by steps 51 us, by rows 45)
    const int from = (s0 + c * U) * 32 + lg * 8;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int u = 0; u < U; ++u) f.w[r][u] = load(wp[r] + from + u * 32);
#pragma unroll
    for (int u = 0; u < U; ++u) f.x[u] = load(xp + from + u * 32);
    if (NORM) {
#pragma unroll
      for (int u = 0; u < U; ++u) f.g[u] = load(a.norm + from + u * 32);
    }
  };
  auto use = [&](const Chunk& f) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      bf16x8_t v = f.x[u];
      if (NORM) v = normed(v, f.g[u]);
#pragma unroll
      for (int r = 0; r < RT; ++r)
        acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[r][u], v, acc[r],
                                                         0, 0, 0);
    }
  };
  static_assert(YT <= NW, "a tile of y for a wave");
  Ends<ACT> ends;
  Chunk one, two;
  if (wid < chunks) fetch(one, wid);
  if (a.fours && wid < YT) ends.read(a, l16, row0 + wid * 16 + lg * 4);
  // fetches under a condition would have their users wait for all that is under way (one
  // of x, 4096 rows of 14336 24.3 us so, 23.7 as it is; 32000 of 2048 with norm 27.0, 26.0)
  int c = wid;
  for (; c + 2 * NW < chunks; c += 2 * NW) {
    fetch(two, c + NW);
    __builtin_amdgcn_sched_barrier(0);
    use(one);
    __builtin_amdgcn_sched_barrier(0);
    fetch(one, c + 2 * NW);
    __builtin_amdgcn_sched_barrier(0);
    use(two);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (c + NW < chunks) {
    fetch(two, c + NW);
    __builtin_amdgcn_sched_barrier(0);
    use(one);
    use(two);
  } else if (c < chunks) {
    use(one);
  }
  // steps that make no whole chunk
  for (int s = s0 + chunks * U + wid; s < s0 + steps; s += NW) {
    const int at = s * 32 + lg * 8;
    bf16x8_t v = load(xp + at);
    if (NORM) v = normed(v, load(a.norm + at));
#pragma unroll
    for (int r = 0; r < RT; ++r)
      acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load(wp[r] + at), v,
                                                       acc[r], 0, 0, 0);
  }

#pragma unroll
  for (int r = 0; r < RT; ++r) red[wid][r][lane] = acc[r];
  if (NORM) squares[wid][lane] = sq;
  __syncthreads();

  if (a.zero && blockIdx.x == 0)
    for (int i = threadIdx.x; i < a.n_zero; i += NW * WAVE) a.zero[i] = 0;
  // a wave per tile of y: four columns of a row a lane
  if (wid < YT) {
    const int r = wid;
    f32x4 v[ACT ? 2 : 1];
#pragma unroll
    for (int h = 0; h < (ACT ? 2 : 1); ++h) {
      v[h] = red[0][r + h * YT][lane];
#pragma unroll
      for (int w = 1; w < NW; ++w) {
        const f32x4 p = red[w][r + h * YT][lane];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[h][j] += p[j];
      }
    }
    if (NORM) {
      float s = 0.0f;
#pragma unroll
      for (int w = 0; w < NW; ++w) s += squares[w][lane];
      s += __shfl_xor(s, 16, WAVE);
      s += __shfl_xor(s, 32, WAVE);
      const float f = rsqrtf(s / a.K + a.eps);
#pragma unroll
      for (int h = 0; h < (ACT ? 2 : 1); ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[h][j] *= f;
    }
    if (SHARED && !sums_of_all(a, (long)blockIdx.x * YT + r, lane, v[0])) return;
    if (l16 < a.M) finish_columns<ACT>(a, l16, row0 + r * 16 + lg * 4, v, ends);
  }
}

// Blocks that share a tile's contraction, as many as have something of it.
// per: steps or stages of a chunk
static dim3 shared_grid(LinearFewArgs& a, int cols, int steps, int per, int split) {
  a.share = (steps + split - 1) / split;
  const int parts = (steps + a.share - 1) / a.share;
  a.parts = (unsigned char)parts;
  const int chunks = a.share / per;
  a.turn = chunks > 1 && in_step(a.ldw)
               ? (unsigned)(((1ull << 32) + chunks - 1) / chunks) : 0;
  return dim3((unsigned)((a.O + cols - 1) / cols), (unsigned)parts);
}

template <int RT, int ACT, int NW, int U>
static void linear_few_go(LinearFewArgs a, int split, hipStream_t stream) {
  constexpr int cols = 16 * (ACT ? RT / 2 : RT);
  // the norm's weights and sums need registers: shorter chunks
  const dim3 grid = shared_grid(a, cols, a.K / 32, a.norm ? 2 : U, split);
  const dim3 block(NW * WAVE);
  if constexpr (RT == 1 && U == 2) {
    if (a.parts > 1) {
      linear_few_kernel<RT, ACT, false, NW, U, true><<<grid, block, 0, stream>>>(a);
      return;
    }
  }
  if (a.norm) {
    linear_few_kernel<RT, ACT, true, NW, 2, false><<<grid, block, 0, stream>>>(a);
  } else {
    linear_few_kernel<RT, ACT, false, NW, U, false><<<grid, block, 0, stream>>>(a);
  }
}

// Tiles of W's rows per block.  A CU reads about 30 bytes a nanosecond, W and, from L2, x,
// so it is those with which the busiest CU reads the fewest rows of both: its blocks, one
// after the other, times what a block reads.  Over 2800 random sizes these are within .4%
// of the fastest (us with one, two, four: 28672 rows of 4096, one of x 38, 42, 45; 16 of x
// 56, 51, 48; 8192 of 3584, 12 of x 15.8, 15.0, 18.2; 11312 of 1472, one of x 8.0, 8.6,
// 9.4).  Through registers a block's norm or unit costs about four rows more, and 24 where
// rows are short; four tiles else three, as they have fewer loads under way (units of one of
// x, 26528 of 512 with two 15.9, four 13.1; 7 of x, norm, 23552 rows of 576 9.9, 8.8; 4 of
// x, 26272 rows of 3840 with one 39.1, four 42.5).  through: rows of x by LDS, up to 8 as 8
// (which has four tiles wherever so few are).
static int few_tiles(int M, int O, int K, int act, bool norm, bool through) {
  const bool more = act || norm;
  const int rows = through ? max(M, 8) : M + (!more ? 0 : K <= 1024 ? 24 : 4);
  int best = 0;
  long least = 0;
  for (int tiles = 4; tiles >= (act ? 2 : 1); tiles /= 2) {
    const int cols = 16 * tiles / (act ? 2 : 1), blocks = (O + cols - 1) / cols;
    const int fewer = tiles == 4 && !more && !through ? 3 : 0;
    const long reads = (long)((blocks + 255) / 256) * (16 * tiles + rows + fewer);
    if (!best || reads < least) best = tiles, least = reads;
  }
  return best;
}

// One tile takes two steps at a time (4096 rows of 4096 8.3 us, of 14336 22.2, with four 9.2
// and 23.3; 23744 rows of 544 7.5, 9.1), but four in long rows of more than one round
// (28672 of 4096 41, 38).
static void linear_few_tiles(const LinearFewArgs& a, int act, int split,
                             hipStream_t stream) {
  const int tiles = few_tiles(a.M, a.O, a.K, act, a.norm != nullptr, false);
  if (act == LF_SILU) {
    if (tiles == 4) linear_few_go<4, LF_SILU, 4, 2>(a, 1, stream);
    else linear_few_go<2, LF_SILU, 8, 4>(a, 1, stream);
  } else if (act == LF_GELU) {
    if (tiles == 4) linear_few_go<4, LF_GELU, 4, 2>(a, 1, stream);
    else linear_few_go<2, LF_GELU, 8, 4>(a, 1, stream);
  } else if (tiles == 4) {
    linear_few_go<4, LF_PLAIN, 4, 2>(a, 1, stream);
  } else if (tiles == 2) {
    linear_few_go<2, LF_PLAIN, 8, 4>(a, 1, stream);
  } else if (a.O > 4096 && a.K >= 4096) {
    linear_few_go<1, LF_PLAIN, 8, 4>(a, 1, stream);
  } else {
    linear_few_go<1, LF_PLAIN, 8, 2>(a, split, stream);
  }
}

// The same for more rows of x (few_through_lds).  Read by each wave from L2 as above, they
// would be the larger part of what is read, and 64 bytes of each of 16 rows take a
// load four times as long as whole lines; here x and W come to LDS in whole lines, KS
// steps of 32 columns at a time, into a ring of stages.  A wave takes one of the steps,
// for all rows of W and of x or for half of x's.
// Measured, beside the library's product (us; M x K x O): 17 x 2048 x 2048: 6.2, 11.0;
// 64 of these: 8.4, 11.7; 64 x 2816 x 2048: 10.0, 14.7; 64 x 2048 x 11264: 15.4, 16.0;
// 64 x 4096 x 4096: 13.7, 15.1; 64 x 4096 x 28672: 54, 51, with norm and unit 59,
// beside 60 for three kernels; 64 x 14336 x 4096: 40, 39.  W to registers by rows of 64
// bytes: 10.6 us for 64 x 2048 x 2048, 70 for 64 x 4096 x 28672.
#define LS_WAVES 8

// What blocks have of a contraction: all of it, from the first column on or, where the memory
// asks for it, from a column of their own (first_of), or a share.  Few blocks gain nothing by
// a column of their own, and what it and shares take cost short kernels up to 8% (17 of x;
// 512 rows of 4096 6.4 us without, 6.8 with, 1024 of 8192 12.7, 12.7, 2048 13.8, 13.25, 4096
// 17.5, 15.4; units of 2048 of 4096 with norm 14.0, 14.3, of 3072 of 8192 26.8, 25.9).
// Four tiles a block are for rows enough.
enum { LS_WHOLE = 0, LS_TURNED = 1, LS_SHARED = 2 };

// RT, TT: tiles of 16 rows of W and of x
template <int RT, int TT, int KS, int ACT, bool NORM, int WAY>
__global__ __launch_bounds__(LS_WAVES * WAVE) void linear_some_kernel(
    const LinearFewArgs a) {
  constexpr int YT = ACT ? RT / 2 : RT;
  constexpr int PARTS = (RT + TT) * KS / LS_WAVES;  // loads to LDS, wave and stage
  constexpr int STAGE = (RT + TT) * KS * 1024;
  constexpr int RING = 4 * STAGE > 140 * 1024 ? 3 : 4;
  // loads of a wave that may be under way when it comes to a stage
  constexpr int BEHIND = (RING - 2) * (PARTS + (NORM ? 1 : 0));
  constexpr int TW = TT * KS / LS_WAVES;            // tiles of x of a wave
  constexpr int RP = KS * 4;                        // pieces of 16 bytes of a row
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ float squares[NORM ? LS_WAVES : 1][TW][WAVE];

  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int l16 = lane & 15, lg = lane >> 4;
  const int step = wid % KS, tile0 = wid / KS * TW;
  const int row0 = blockIdx.x * 16 * YT;

  // A load to LDS is 1 KB of rows of W, then of x.  Pieces of a row are swapped by the
  // row: those that a read meets lie in different banks.
  auto place = [](int row, int piece) { return piece ^ (row & 15); };
  const char* from[PARTS];
  int col[PARTS];
#pragma unroll
  for (int i = 0; i < PARTS; ++i) {
    const int at = (i * LS_WAVES + wid) * WAVE + lane, row = at / RP;
    col[i] = place(row, at % RP) * 8;
    if (row < RT * 16) {
      const int r = row / 16 / YT * a.O + min(row0 + row / 16 % YT * 16 + row % 16, a.O - 1);
      from[i] = (const char*)(a.w + (long)r * a.ldw);
    } else {
      from[i] = (const char*)(a.x + (long)min(row - RT * 16, a.M - 1) * a.ldx);
    }
  }
  bf16x8_t g[NORM ? RING : 1];
  constexpr int W = KS * 32;  // columns of a stage
  const int s0 = WAY == LS_SHARED ? blockIdx.y * a.share : 0;
  const int all = (a.K + W - 1) / W - s0;
  const int stages = WAY == LS_SHARED ? min(a.share, all) : all;
  // the first column of a stage, counted from those that the loop is at.  Stages behind the
  // last one repeat it, and columns behind the last one others of its row; nobody takes
  // them (64 of x, 28672 rows of 4096 with norm 53.6 us, 54.4 where they are the first again)
  const int end = (s0 + stages) * W, span = stages * W;
  int base = (s0 + (WAY == LS_WHOLE ? 0 : first_of(a, a.share, stages, blockIdx.x))) * W;
  const int last = base + span - W;
  auto column = [&](int t) {
    int k = base + t * W;
    if (WAY == LS_WHOLE) return k;
    k = min(k, last);
    return k >= end ? k - span : k;
  };
  auto issue = [&](int t, int slot) {
    const int k0 = column(t);
#pragma unroll
    for (int i = 0; i < PARTS; ++i)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(
              from[i] + (unsigned)min(k0 + col[i], a.K - 8) * 2),
          (__attribute__((address_space(3))) void*)(
              smem + slot * STAGE + (i * LS_WAVES + wid) * 1024), 16, 0, 0);
    if (NORM)
      g[slot] = *reinterpret_cast<const bf16x8_t*>(
          a.norm + min(k0 + step * 32, a.K - 32) + lg * 8);
  };
  f32x4 acc[RT][TW];
  float sq[TW];
#pragma unroll
  for (int i = 0; i < TW; ++i) {
    sq[i] = 0.0f;
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[r][i] = f32x4{0, 0, 0, 0};
  }
  auto use = [&](int s) {
    if (column(s) + step * 32 >= a.K) return;
    const char* at = smem + s * STAGE + l16 * RP * 16 + place(l16, step * 4 + lg) * 16;
    bf16x8_t w[RT], v[TW];
#pragma unroll
    for (int r = 0; r < RT; ++r)
      w[r] = *reinterpret_cast<const bf16x8_t*>(at + r * RP * 256);
#pragma unroll
    for (int i = 0; i < TW; ++i)
      v[i] = *reinterpret_cast<const bf16x8_t*>(at + (RT + tile0 + i) * RP * 256);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < TW; ++i) {
      if (NORM) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float f = (float)v[i][j];
          sq[i] = fmaf(f, f, sq[i]);
          v[i][j] = (__bf16)(f * ((float)g[s][j] + a.offset));
        }
      }
#pragma unroll
      for (int r = 0; r < RT; ++r)
        acc[r][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[r], v[i], acc[r][i],
                                                            0, 0, 0);
    }
  };
#pragma unroll
  for (int t = 0; t < RING - 1; ++t) issue(t, t);
  // younger than what the first stages wait for: they wait for no less
  constexpr int TILES = (YT * TT + LS_WAVES - 1) / LS_WAVES;  // of y and x, of a wave
  Ends<ACT> ends[TILES];
#pragma unroll
  for (int q = 0; q < TILES; ++q) {
    const int n = min(wid + q * LS_WAVES, YT * TT - 1);
    if (a.fours) ends[q].read(a, n % TT * 16 + l16, row0 + n / TT * 16 + lg * 4);
  }
  int t0 = 0;
  for (; t0 + RING <= stages; t0 += RING) {
#pragma unroll
    for (int s = 0; s < RING; ++s) {
      __builtin_amdgcn_sched_barrier(0);
      // vmcnt, in a form that the compiler takes into account
      __builtin_amdgcn_s_waitcnt((BEHIND & 15) | (BEHIND >> 4) << 14 | 0xf70);
      asm volatile("s_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      issue(s + RING - 1, (s + RING - 1) % RING);
      use(s);
    }
    base += RING * W;
  }
  // the remainder is on its way
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0xf70 & ~0xc00f);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int s = 0; s < RING - 1; ++s)
    if (t0 + s < stages) use(s);
  __syncthreads();
  f32x4* red = reinterpret_cast<f32x4*>(smem);  // [steps][RT][TT][lanes]
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int i = 0; i < TW; ++i)
      red[((step * RT + r) * TT + tile0 + i) * WAVE + lane] = acc[r][i];
  if (NORM) {
#pragma unroll
    for (int i = 0; i < TW; ++i) squares[wid][i][lane] = sq[i];
  }
  __syncthreads();

  if (a.zero && blockIdx.x == 0)
    for (int i = threadIdx.x; i < a.n_zero; i += LS_WAVES * WAVE) a.zero[i] = 0;
#pragma unroll
  for (int q = 0; q < TILES; ++q) {
    const int n = wid + q * LS_WAVES, r = n / TT, i = n % TT;
    if (n >= YT * TT) break;
    f32x4 v[ACT ? 2 : 1];
#pragma unroll
    for (int h = 0; h < (ACT ? 2 : 1); ++h) {
      v[h] = f32x4{0, 0, 0, 0};
#pragma unroll
      for (int q = 0; q < KS; ++q) {
        const f32x4 p = red[((q * RT + r + h * YT) * TT + i) * WAVE + lane];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[h][j] += p[j];
      }
    }
    if (NORM) {
      float s = 0.0f;
#pragma unroll
      for (int q = 0; q < KS; ++q) s += squares[i / TW * KS + q][i % TW][lane];
      s += __shfl_xor(s, 16, WAVE);
      s += __shfl_xor(s, 32, WAVE);
      const float f = rsqrtf(s / a.K + a.eps);
#pragma unroll
      for (int h = 0; h < (ACT ? 2 : 1); ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[h][j] *= f;
    }
    if (WAY == LS_SHARED &&
        !sums_of_all(a, ((long)blockIdx.x * YT + r) * TT + i, lane, v[0]))
      continue;
    if (i * 16 + l16 < a.M)
      finish_columns<ACT>(a, i * 16 + l16, row0 + r * 16 + lg * 4, v, ends[q]);
  }
}

template <int RT, int TT, int ACT, bool NORM>
static void linear_some_go(LinearFewArgs a, int split, hipStream_t stream) {
  constexpr int KS = RT == 1 ? 8 : 4;
  constexpr int cols = 16 * (ACT ? RT / 2 : RT);
  constexpr int stage = (RT + TT) * KS * 1024;
  constexpr int ring = (4 * stage > 140 * 1024 ? 3 : 4) * stage;
  constexpr int smem = ring > KS * RT * TT * 1024 ? ring : KS * RT * TT * 1024;
  const dim3 grid = shared_grid(a, cols, (a.K + KS * 32 - 1) / (KS * 32), 1, split);
  auto go = [&](auto kernel) {
    if (smem > 56 * 1024)  // with the sums of squares above the default limit
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    kernel<<<grid, dim3(LS_WAVES * WAVE), smem, stream>>>(a);
  };
  if constexpr (RT > 1 && !ACT && !NORM) {
    if (a.parts > 1) return go(&linear_some_kernel<RT, TT, KS, ACT, NORM, LS_SHARED>);
  }
  if (a.turn && (RT == 4 || grid.x >= (ACT || NORM ? 192 : 128)))
    go(&linear_some_kernel<RT, TT, KS, ACT, NORM, LS_TURNED>);
  else
    go(&linear_some_kernel<RT, TT, KS, ACT, NORM, LS_WHOLE>);
}

template <int RT, int ACT>
static void linear_some_tiles(const LinearFewArgs& a, int split, hipStream_t stream) {
  if (a.M <= 32) {
    if (a.norm) {
      linear_some_go<RT, 2, ACT, true>(a, split, stream);
    } else {
      linear_some_go<RT, 2, ACT, false>(a, split, stream);
    }
  } else {
    if (a.norm) {
      linear_some_go<RT, 4, ACT, true>(a, split, stream);
    } else {
      linear_some_go<RT, 4, ACT, false>(a, split, stream);
    }
  }
}

// Blocks that share a contraction have two tiles up to 2048 rows and four above (few_split).
static void linear_some(const LinearFewArgs& a, int act, int split, hipStream_t stream) {
  const int tiles = split > 1 ? (a.O <= 2048 ? 2 : 4)
                              : few_tiles(a.M, a.O, a.K, act, a.norm != nullptr, true);
  if (act == LF_SILU) {
    if (tiles == 4) linear_some_tiles<4, LF_SILU>(a, 1, stream);
    else linear_some_tiles<2, LF_SILU>(a, 1, stream);
  } else if (act == LF_GELU) {
    if (tiles == 4) linear_some_tiles<4, LF_GELU>(a, 1, stream);
    else linear_some_tiles<2, LF_GELU>(a, 1, stream);
  } else if (tiles == 1) {
    linear_some_tiles<1, LF_PLAIN>(a, 1, stream);
  } else if (tiles == 2) {
    linear_some_tiles<2, LF_PLAIN>(a, split, stream);
  } else {
    linear_some_tiles<4, LF_PLAIN>(a, split, stream);
  }
}

// Whether rows of x go through LDS: above 16, and fewer where rows are long, as a block's
// chain through registers is the longer one.  Time by LDS over that by registers: 9 to 16 of
// x, rows of 2304 to 4096 .63 to 1.04, of 2048 .84 to 1.02 for 8192 to 12288 rows of W (16 of
// x without a norm .95 to .97 from 4096 on) and up to 1.24 for others; into up to 4096 with
// norm, 9 of x 1.08 to 1.17, 12 1.02 to 1.11, 16 of 4096 .97 to 1.0 and of 8192 .9; up to 8
// of x, with a norm or unit, 8192 to 12288 rows of W of 2304 and more .87 to 1.03, others 1.0
// to 1.35.
static bool few_through_lds(int M, int O, int K, int act, bool norm) {
  const int rows = (act ? 2 : 1) * O;
  const bool some = rows > (M > 12 && !norm ? 4096 : 8192) && rows <= 12288;
  if (M > 16) return true;
  if (M <= 8) return (act || norm) && K > 2048 && some;
  if (norm && !act && rows <= 4096) return M > 12 && K >= 4096;
  return K > 2048 || (K == 2048 && some);
}

// Blocks that share a tile's contraction where the caller has room for their sums, as many
// as come in one round: x is read once per block, four times W with 16 rows of W and 64 of
// x, so that long rows have blocks of more rows and a part of the columns each, and up to
// 2048 rows of W leave CUs idle without (us, alone and shared: 64 of x, 2048 rows of 8192
// 20.7, 13.4, 4096 of 14336 39.6, 29.0; one of x, 2048 of 8192 11.6, 9.7).  In two rounds
// it loses (64 of x, 2816 rows of 4096 17.4, 19.9; one of x, 2816 of 8192 15.3, 18.3), and
// short rows of more than 16 of x are linear_own_kernel's (shared and there: 64 of x, 1536 rows
// of 2816 7.4, 5.8, 1616 of 4288 10.2, 9.5, 1504 of 5632 10.9, 11.3, 2048 of 8704 16.7, 19.1;
// 20 of x, 1536 of 5120 8.7, 7.9, 29 of x, 2048 of 9216 12.7, 15.3).  With four tiles
// up to 16 of x gain from rows of 12288 into up to 3584 on (12 of x, into 2816 23.8, 21.0,
// into 3584 26.1, 24.3; into 4096 27.7, 28.3; 10240 into 2816 20.6, 20.9).
static int few_split(int M, int O, int K, int act, bool norm) {
  if (act || norm) return 1;
  if (!few_through_lds(M, O, K, act, norm)) return O <= 2048 && K >= 4096 ? 2 : 1;
  if (O <= 2048) return K >= (M > 32 ? 5632 : M > 16 ? 7168 : 4096) ? 4 : 1;
  return K >= 8192 && (M > 16 ? O <= 4096 : K >= 12288 && O <= 3584) ? 4 : 1;
}

// Room for a shared contraction: `numbers` to be cleared before, and sums behind them.
extern "C" long linear_few_room(int M, int O, int K, int* numbers) {
  const int split = few_split(M, O, K, 0, false);
  const int tiles = (O + 63) / 64 * 4 * (M <= 16 ? 2 : (M + 31) / 32 * 2);
  *numbers = split > 1 ? tiles : 0;
  return (long)*numbers * split * WAVE * 4;
}

// Strides in elements; 16-byte loads: x, w, norm and the strides of x and w are
// multiples of 8 elements, K of 32.  M up to 64.  count, part: room for a shared
// contraction, or null; zero: n_zero numbers to clear for one behind this.
extern "C" void launch_linear_few(const void* x, const void* w, const void* bias,
                                  const void* res, const void* norm, void* y,
                                  int M, int O, int K, long ldx, long ldw,
                                  long ldr, long ldy, float eps, float offset,
                                  int act, unsigned* count, float* part,
                                  unsigned* zero, int n_zero, hipStream_t stream) {
  LinearFewArgs a{};
  a.x = (const __bf16*)x, a.w = (const __bf16*)w, a.bias = (const __bf16*)bias;
  a.res = (const __bf16*)res, a.norm = (const __bf16*)norm, a.y = (__bf16*)y;
  a.M = (short)M, a.O = O, a.K = K;
  a.ldx = ldx, a.ldw = ldw, a.ldr = ldr, a.ldy = ldy;
  if (norm) a.eps = eps, a.offset = offset;
  else a.part = part;
  a.count = count, a.zero = zero, a.n_zero = n_zero;
  a.fours = (bias || res) && O % 4 == 0 && (long)bias % 8 == 0 && (long)res % 8 == 0 &&
            (!res || ldr % 4 == 0);
  const int split = count ? few_split(M, O, K, act, norm != nullptr) : 1;
  if (split == 1 && linear_own_go(a, act, stream)) return;
  if (few_through_lds(M, O, K, act, norm != nullptr)) {
    linear_some(a, act, split, stream);
  } else {
    linear_few_tiles(a, act, split, stream);
  }
}
