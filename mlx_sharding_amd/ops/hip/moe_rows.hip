// Routed experts of a decoding step, up to 128 tokens and 64 experts.
//
//   moe_route    residual update, RMS norm, router product, softmax and choice of
//                a token, a block each
//   moe_up       act(gate) * up of every chosen (token, expert) pair
//   moe_down     the pairs' outputs, weighted, in 32 bits
//   moe_combine  a token's pairs, shared experts and residual added up
//
// (9 to 64 tokens with a shared feed-forward, and fewer with a large one, have moe_shared.hip's
// for the first and last)
//
// No sort: a block counts every expert's pairs, which tells its share of the work, and
// looks through the choices (at most 1024) for those of an expert.  Rows of pairs lie at
// token * top + place.
//
// The products are bound by reading the experts' packed weights.  Read naively,
// rows of x out of L2 are twice those bytes and more (16 rows of 16 bits for 16
// rows of 4), which held the kernel before this at 2.7 TB/s.  So rows of x stay
// in registers: a wave of eight takes every eighth unit of 128 of the contraction
// and keeps those parts of 16 tokens while the block walks over its rows of
// weights, the next 16 rows asked for before these are used.  The waves add up
// through LDS.
//
// Within a unit a lane has 32 consecutive values of a row: k = unit * 128 +
// (lane >> 4) * 32 + step * 8 + j, which is 16 bytes at 4 bits and one scale; A
// and B agree on that order.  moe_pack lays packed weights out in it once, a
// tile's scales behind its words: a wave's load is 1 KB in one piece, where rows
// as they come are 64 bytes each and scales 2 (64 tokens, 64 experts of 1408 x
// 2048 at 4 bits: 113 us so, 89 packed).
// 4 and 8 bits become fp16 numbers 1024 + q by an OR, exactly, and one fma rounds
// them to s q + b; values of a word are laid out in pairs for it.  The vector units are
// at work for half of the time at 4 bits; with every second value left where it is, as
// part of 64 + q, and both masks in one instruction a word of eight takes 13 of them
// instead of 19 (64 tokens, both products: 92 -> 87 us).  A wave has one tile's loads under
// way beside the one it works on, and waits for its oldest only (both products 84 -> 71 us).
// Measured, norm, router, choice, experts and sum of 64 experts of 1408 x 2048 (6 a
// token) beside the kernels before (norm and residual apart): 1 token at 4 bits
// 33 us, 48 and norms; 64 tokens 105, 166 (experts alone 3.5 TB/s); 8 bits 147,
// 247; bf16, experts alone, 64 tokens 234 us (4.7 TB/s).

#include "moe_rows.h"
#include "moe_choice.h"

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define MR_WAVES 8
#define MR_BLOCK (MR_WAVES * WAVE)
#define MR_UNIT 128

// -- operands ---------------------------------------------------------------

template <int BITS>
struct Operand {
  typedef f16x8 V;
  typedef f16x4 H;
  typedef _Float16 E;
  static __device__ __forceinline__ f32x4 mma(V a, V b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Operand<16> {
  typedef bf16x8_t V;
  typedef bf16x4_t H;
  typedef __bf16 E;
  static __device__ __forceinline__ f32x4 mma(V a, V b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

// (word & mask) | high in one instruction: with two literals the compiler takes two
__device__ __forceinline__ unsigned masked(unsigned word, unsigned mask, unsigned high) {
  unsigned v;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(v) : "v"(word), "s"(mask), "v"(high));
  return v;
}

// a lane's 32 values of one unit, as they come from memory
template <int BITS>
struct Packed {
  uint4 q[BITS / 4];
  unsigned scale;  // scale and offset, bf16
  // w: this lane's first 16 bytes; sc: its scale (packed only)
  __device__ __forceinline__ void load(const char* w, const char* sc) {
#pragma unroll
    for (int i = 0; i < BITS / 4; ++i)
      q[i] = *reinterpret_cast<const uint4*>(w + i * (BITS == 16 ? 16 : 1024));
    if (BITS < 16) scale = *reinterpret_cast<const unsigned*>(sc);
  }
  // values 8 i .. 8 i + 7
  __device__ __forceinline__ typename Operand<BITS>::V operand(int i) const {
    const unsigned* u = reinterpret_cast<const unsigned*>(q);
    if constexpr (BITS == 16) {
      return __builtin_bit_cast(bf16x8_t, q[i]);
    } else {
      constexpr float MID = BITS == 4 ? 8.0f : 128.0f;
      const float sf = __uint_as_float(scale << 16);
      const _Float16 sh = (_Float16)sf;
      const _Float16 bh = (_Float16)(__uint_as_float(scale & 0xFFFF0000u) + MID * sf);
      const f16x2 s2 = {sh, sh}, b2 = {bh, bh};
      // values as the last bits of 1024 + q, or, four bits up, of 64 + q; from there
      // exactly to q - MID
      constexpr unsigned LOW = BITS == 4 ? 0x000F000Fu : 0x00FF00FFu;
      f16x8 out;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool up = BITS == 4 && (j & 1);
        const unsigned word = BITS == 4 ? u[i] >> (8 * (j / 2))
                                        : u[2 * i + j / 2] >> (8 * (j & 1));
        // (of 8 bits the compiler's two are the faster ones: one token, 8 experts of 512 x
        // 1024 5.9 us, 5.6 so)
        const unsigned v =
            BITS == 8 ? (word & LOW) | 0x64006400u
                      : masked(word, up ? LOW << 4 : LOW, up ? 0x54005400u : 0x64006400u);
        const _Float16 c = (_Float16)((up ? -64.0f : -1024.0f) - MID);
        const f16x2 f =
            (__builtin_bit_cast(f16x2, v) + f16x2{c, c}) * s2 + b2;
        out[2 * j] = f[0];
        out[2 * j + 1] = f[1];
      }
      return out;
    }
  }
};

// -- products ---------------------------------------------------------------

// A tile of the shared feed-forward for up to 8 tokens: the waves take the contraction by
// turns in steps of 64 (two loads of a row, one line of 128 bytes).  Bound by what a CU
// reads, about 30 bytes a nanosecond, so every tile has a block (one token, with 16, 32,
// 64, 128, 176 blocks of 176 tiles beside the experts': 126, 70, 41, 32, 26 us; after
// them 34, as two kernels).  More tokens need the blocks for experts: 16 alone 81 us, so 85.
template <bool UP>
__device__ __forceinline__ void dense_tiles(const MoeRowsArgs& a, f32x4* red) {
  constexpr int MATS = UP ? 2 : 1;
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int l16 = lane & 15, lg = lane >> 4;
  auto load = [](const __bf16* p) { return *reinterpret_cast<const bf16x8_t*>(p); };
  // places within x and w in 32 bits (sizes are up to 4096): pointers were one register
  // too many
  const unsigned xp = min(l16, a.N - 1) * a.DK + lg * 8;
  const int t = blockIdx.x;
  unsigned wp[MATS];
  f32x4 acc[MATS];
#pragma unroll
  for (int m = 0; m < MATS; ++m) {
    wp[m] = (unsigned)(m * a.DO + t * 16 + l16) * a.DK + lg * 8;
    acc[m] = f32x4{0, 0, 0, 0};
  }
  // three ahead: what a wave has of 2048 columns is four
  constexpr int AHEAD = 4;
  struct Part {
    bf16x8_t w[MATS][2], x[2];
  } part[AHEAD];
  auto fetch = [&](Part& f, int k) {
    if (k >= a.DK) return;
#pragma unroll
    for (int m = 0; m < MATS; ++m)
#pragma unroll
      for (int i = 0; i < 2; ++i) f.w[m][i] = load(a.dw + (wp[m] + k + i * 32));
#pragma unroll
    for (int i = 0; i < 2; ++i) f.x[i] = load(a.dx + (xp + k + i * 32));
  };
  constexpr int STEP = MR_WAVES * 64;
#pragma unroll
  for (int p = 0; p < AHEAD - 1; ++p) fetch(part[p], wid * 64 + p * STEP);
  for (int k = wid * 64; k < a.DK; k += AHEAD * STEP) {
#pragma unroll
    for (int p = 0; p < AHEAD; ++p) {
      if (k + p * STEP >= a.DK) break;
      fetch(part[(p + AHEAD - 1) % AHEAD], k + (p + AHEAD - 1) * STEP);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int m = 0; m < MATS; ++m)
          acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(part[p].w[m][i],
                                                           part[p].x[i], acc[m], 0, 0, 0);
    }
  }
#pragma unroll
  for (int m = 0; m < MATS; ++m) red[(wid * MATS + m) * WAVE + lane] = acc[m];
  __syncthreads();
  if (wid != 0 || l16 >= a.N) return;
  f32x4 v[MATS];
#pragma unroll
  for (int m = 0; m < MATS; ++m) {
    v[m] = red[m * WAVE + lane];
#pragma unroll
    for (int w = 1; w < MR_WAVES; ++w) {
      const f32x4 p = red[(w * MATS + m) * WAVE + lane];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[m][j] += p[j];
    }
  }
  bf16x4_t h;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float g = v[0][j];
    h[j] = (__bf16)(UP ? g / (1.0f + __expf(-g)) * v[MATS - 1][j] : g);
  }
  *reinterpret_cast<bf16x4_t*>(a.dy + (long)l16 * a.DO + t * 16 + lg * 4) = h;
}

// Work is counted in tiles: 16 rows of an expert's matrices by up to 16 of its pairs.
// Every block counts the pairs of all experts and takes an even share of all tiles, one
// after the other.  With a block per expert and range of rows the longest one has the
// expert with most pairs (both products of 64 experts of 1408 x 2048 at 4 bits: 64 tokens
// 94.9 us so, 86.9 shared; 128 130.7, 95.9; one, whose choices are counted first, 19.8,
// 17.5).  Choices stay in LDS for the search of an expert's pairs, which goes through
// them one load after the other otherwise (64 tokens, both products: 97 us from memory,
// 92 so).  Up to 64 pairs are a lane each of one wave, which finds those of an expert by
// ballots (one token 19.4 us by counts in LDS, 17.5 so; 32 pairs of 64 experts of 256 x
// 512 10.9 and, with shares that end with a group, 8.7; a block per expert 8.1).  What
// that is slower than a block per expert, up to 1 us for both products of small experts,
// is the counting.
template <int BITS, int UPW, bool UP>
constexpr bool two_a_cu() {
  return UPW <= (BITS == 16 && UP ? 1 : 2);
}

// FEW: up to 64 pairs
template <int BITS, int GS, int UPW, bool UP, bool FEW>
__global__ __launch_bounds__(
    MR_BLOCK, (two_a_cu<BITS, UPW, UP>() ? 4 : 2)) void moe_rows_kernel(
    const MoeRowsArgs a) {
  typedef Operand<BITS> Op;
  typedef typename Op::V V;
  constexpr int MATS = UP ? 2 : 1;
  __shared__ int count[64], ends[64];
  __shared__ unsigned long long members[FEW ? 64 : 1];  // of the pairs, those of an expert
  __shared__ short list[16];
  __shared__ unsigned char chosen[FEW ? 1 : MR_PAIRS];  // experts, 255: none
  __shared__ __attribute__((aligned(16))) f32x4 red[2][MR_WAVES][MATS][WAVE];

  if ((int)blockIdx.x < a.dense) {
    dense_tiles<UP>(a, &red[0][0][0][0]);
    return;
  }
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int l16 = lane & 15, lg = lane >> 4;
  const int rows = a.O / 16;
  // of the lanes up to this one the sum of (n + 15) / 16, which is below 2^PLANES: groups
  // of pairs up to a lane's expert
  auto groups_up_to = [&](int n) {
    constexpr int PLANES = FEW ? 3 : 7;
    const unsigned long long upto = ~0ull >> (WAVE - 1 - lane);
    const int g = (n + 15) / 16;
    int sum = 0;
#pragma unroll
    for (int b = 0; b < PLANES; ++b) sum += __popcll(__ballot(g >> b & 1) & upto) << b;
    return sum;
  };
  // An entry per expert; FEW: per pair, of which the first of its expert counts, and what
  // it holds comes by ballots of one wave.
  if constexpr (FEW) {
    if (wid == 0) {
      const unsigned e = lane < a.pairs ? a.choice[lane] : 255u;
      unsigned long long same = __ballot(e < (unsigned)a.experts);
#pragma unroll
      for (int b = 0; b < 6; ++b) {
        const bool bit = e >> b & 1;
        const unsigned long long with = __ballot(bit);
        same &= bit ? with : ~with;
      }
      const bool leads = e < (unsigned)a.experts && __ffsll(same) - 1 == lane;
      ends[lane] = groups_up_to(leads ? __popcll(same) : 0);
      count[lane] = e;
      members[lane] = same;
    }
  } else {
    if (threadIdx.x < 64) count[threadIdx.x] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < a.pairs; i += MR_BLOCK) {
      const unsigned e = a.choice[i];
      chosen[i] = (unsigned char)min(e, 255u);
      if (e < (unsigned)a.experts) atomicAdd(&count[e], 1);
    }
    __syncthreads();
    if (wid == 0) ends[lane] = groups_up_to(count[lane]);
  }
  __syncthreads();
  const unsigned groups = __builtin_amdgcn_readfirstlane(ends[WAVE - 1]), all = groups * rows;
  // This block's share of them.  `per` is the largest share that there has to be: with as
  // many rows to every block of a group, and fewer to its last one, where that takes no more
  // blocks, so that no block begins twice; else all / blocks or one more, from 0 to `all`
  // over all blocks.  Divisions are multiplications by reciprocals: exact ones, but that of
  // the last way.
  auto over = [](unsigned x, unsigned n) {  // below 2^16
    return (unsigned)(((float)x + 0.5f) * __builtin_amdgcn_rcpf((float)n));
  };
  const unsigned b = blockIdx.x - a.dense, blocks = gridDim.x - a.dense;
  const unsigned per = max(1u, __umulhi(all + blocks - 1, a.by_blocks));
  const unsigned parts = over(rows + per - 1, per);
  int at, stop;
  if (groups * parts <= blocks) {
    const unsigned group = over(b, parts);
    at = min(group, groups) * rows + (b - group * parts) * per;
    stop = group < groups ? min((group + 1) * rows, at + per) : at;
  } else {
    at = __umulhi(b * all, a.by_blocks);
    stop = __umulhi((b + 1) * all, a.by_blocks);
  }

  const int units = a.K / MR_UNIT;
  const int k0 = wid * MR_UNIT + lg * 32;
  constexpr int UNIT = (16 * MR_UNIT * BITS / 32 + 16 * (MR_UNIT / GS)) * 4;
  const long step = BITS == 16 ? (long)16 * a.K * 2 : (long)units * UNIT;
  const int scales = 16 * MR_UNIT * BITS / 8 - lane * 16 +
                     (l16 * (MR_UNIT / GS) + lg * 32 / GS) * 4;
  int buf = 0;
  while (at < stop) {
    // What follows from a lane's number is made anew for each group of more than 64 pairs in
    // bf16 with one unit a wave: kept, it is more than there are registers for, and reloads
    // wait for the words that are under way (64 tokens, top 6 of 64 experts of 1024 x 1024:
    // 93.0 us, 84.2 so; with loads that products wait for 87.4).
    int self = lane;
    if constexpr (BITS == 16 && UPW == 1 && !FEW) asm volatile("" : "+v"(self));
    const int l16 = self & 15, lg = self >> 4;
    // one group of one expert's pairs, rows t0 to t1
    const int group = __umulhi(at, a.by_rows), t0 = at - group * rows;
    const int t1 = min(rows, t0 + stop - at);
    at += t1 - t0;
    const int place = __popcll(__ballot(ends[lane] <= group));
    auto same = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    const int first = (group - (place ? same(ends[place - 1]) : 0)) * 16;
    const int e = FEW ? same(count[place]) : place;
    const int n = min(16, same(FEW ? __popcll(members[place]) : count[place]) - first);

    // this lane's place in its first unit of the first rows
    const long begin = ((long)e * rows + t0) * step +
                       (BITS == 16 ? ((long)l16 * a.K + k0) * 2
                                   : (long)wid * UNIT + lane * 16);
    const char* wp[2] = {(const char*)a.w + begin, (const char*)a.w2 + begin};
    auto fetch = [&](Packed<BITS>& r, int m, int u, int t) {
      constexpr int far = MR_WAVES * (BITS == 16 ? MR_UNIT * 2 : UNIT);
      const char* p = wp[m] + t * step + (long)u * far;  // between a wave's units
      r.load(p, p + scales);
    };
    // C units of this wave.  Their number is known: where loads are left out between
    // others, the compiler has more waited for than is used (both products of 64 tokens at
    // 4 bits, 64 experts: 84.5 us, 71.5 so; 1 token 16.9, 15.5; 64 at 8 bits 127, 119, in
    // bf16 227, 221).
    auto work = [&](auto mine, auto has) {
      constexpr int C = decltype(mine)::value;
      Packed<BITS> next[MATS][C];
#pragma unroll
      for (int u = 0; u < C; ++u) {
        if (!has(u)) continue;
#pragma unroll
        for (int m = 0; m < MATS; ++m) fetch(next[m][u], m, u, 0);
      }
      int pair;
      if constexpr (FEW) {
        // the n pairs from `first` on go to the lowest lanes, the others anywhere else
        const unsigned long long which = members[place];
        const int to = __popcll(which & ((1ull << self) - 1)) - first;
        const bool listed = (which >> self & 1) && to >= 0 && to < 16;
        pair = __builtin_amdgcn_ds_permute((listed ? to : 16 + self % 48) * 4, lane);
        pair = __shfl(pair, min(l16, n - 1), WAVE);
      } else {
        if (wid == 0) {
          int found = -first;
          for (int i = 0; i < a.pairs && found < 16; i += WAVE) {
            const bool mine = i + self < a.pairs && chosen[i + self] == e;
            const unsigned long long with = __ballot(mine);
            const int place = found + __popcll(with & ((1ull << self) - 1));
            if (mine && place >= 0 && place < 16) list[place] = (short)(i + self);
            found += __popcll(with);
          }
        }
        __syncthreads();
        pair = list[min(l16, n - 1)];
      }
      // asked for here: behind the products it was waited for
      const float weight = UP ? 0.0f : a.weight[pair];
      V x[C][4];
#pragma unroll
      for (int u = 0; u < C; ++u) {
        if (!has(u)) continue;
        const short* src = (const short*)a.x +
                           (long)(UP ? pair / a.top : pair) * a.K + k0 +
                           u * MR_WAVES * MR_UNIT;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (UP && BITS != 16) {
            const bf16x8_t v = *reinterpret_cast<const bf16x8_t*>(src + i * 8);
#pragma unroll
            for (int j = 0; j < 8; ++j) x[u][i][j] = (_Float16)(float)v[j];
          } else {
            x[u][i] = *reinterpret_cast<const V*>(src + i * 8);
          }
        }
      }
      for (int t = t0; t < t1; ++t, buf ^= 1) {
        f32x4 acc[MATS];
#pragma unroll
        for (int m = 0; m < MATS; ++m) acc[m] = f32x4{0, 0, 0, 0};
        const int ahead = min(t + 1, t1 - 1) - t0;
#pragma unroll
        for (int u = 0; u < C; ++u) {
          if (!has(u)) continue;
#pragma unroll
          for (int m = 0; m < MATS; ++m) {
            // The next words come into the registers that are free after these products: a
            // copy of a load that is under way would wait for it.
#pragma unroll
            for (int i = 0; i < 4; ++i)
              acc[m] = Op::mma(next[m][u].operand(i), x[u][i], acc[m]);
            __builtin_amdgcn_sched_barrier(0);
            fetch(next[m][u], m, u, ahead);
          }
        }
#pragma unroll
        for (int m = 0; m < MATS; ++m) red[buf][wid][m][self] = acc[m];
        __syncthreads();
        // one wave finishes these rows, the others go on
        if (wid != t % MR_WAVES) continue;
        f32x4 v[MATS];
#pragma unroll
        for (int m = 0; m < MATS; ++m) {
          v[m] = red[buf][0][m][self];
#pragma unroll
          for (int w = 1; w < MR_WAVES; ++w) {
            const f32x4 p = red[buf][w][m][self];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[m][j] += p[j];
          }
        }
        if (l16 >= n) continue;
        const long to = (long)pair * a.O + t * 16 + lg * 4;
        if constexpr (UP) {
          typedef typename Op::H H4;
          H4 h;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float g = v[0][j];
            h[j] = (typename Op::E)(g / (1.0f + __expf(-g)) * v[MATS - 1][j]);
          }
          *reinterpret_cast<H4*>((typename Op::E*)a.y + to) = h;
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) v[0][j] *= weight;
          *reinterpret_cast<f32x4*>((float*)a.y + to) = v[0];
        }
      }
    };
    // UPW is units / MR_WAVES, rounded up (the launch has an instance for each), so a wave
    // has UPW of them or one less, and without a second one maybe none.
    auto there = [&](int u) { return wid + u * MR_WAVES < units; };
    auto always = [](int) { return true; };
    if constexpr (UPW == 1) work(std::integral_constant<int, UPW>(), there);
    else if (there(UPW - 1)) work(std::integral_constant<int, UPW>(), always);
    else work(std::integral_constant<int, UPW - 1>(), always);
  }
}

// A wave per tile of 16 rows by one unit: words in operand order, pairs of values
// 16 bits apart, then (scale, offset) of every row and group.
template <int BITS>
__global__ __launch_bounds__(WAVE) void moe_pack_kernel(
    const unsigned* __restrict__ w, const unsigned short* __restrict__ scale,
    const unsigned short* __restrict__ offset, unsigned* __restrict__ out, int K,
    int gs, int words) {
  const int units = K / MR_UNIT;
  const long tile = blockIdx.x / units;
  const int unit = blockIdx.x % units;
  const int lane = threadIdx.x, l16 = lane & 15, lg = lane >> 4;
  const long row = tile * 16 + l16;
  unsigned* dst = out + (long)blockIdx.x * words;
  const unsigned* src = w + row * (K * BITS / 32) +
                        (unit * MR_UNIT + lg * 32) * BITS / 32;
#pragma unroll
  for (int i = 0; i < BITS / 4; ++i) {
    const uint4 q = *reinterpret_cast<const uint4*>(src + i * 4);
    uint4 r;
    const unsigned* a = reinterpret_cast<const unsigned*>(&q);
    unsigned* b = reinterpret_cast<unsigned*>(&r);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const unsigned v = a[j];
      if (BITS == 4) {
        const unsigned even = (v & 0xF) | (v >> 4 & 0xF0) | (v >> 8 & 0xF00) |
                              (v >> 12 & 0xF000);
        const unsigned u = v >> 4;
        const unsigned odd = (u & 0xF) | (u >> 4 & 0xF0) | (u >> 8 & 0xF00) |
                             (u >> 12 & 0xF000);
        b[j] = even | odd << 16;
      } else {
        b[j] = (v & 0xFF0000FFu) | (v >> 8 & 0xFF00) | (v << 8 & 0xFF0000);
      }
    }
    *reinterpret_cast<uint4*>(dst + i * 256 + lane * 4) = r;
  }
  const int groups = MR_UNIT / gs;
  for (int i = lane; i < 16 * groups; i += WAVE) {
    const long at = (tile * 16 + i / groups) * (K / gs) + unit * groups + i % groups;
    dst[16 * MR_UNIT * BITS / 32 + i] = scale[at] | (unsigned)offset[at] << 16;
  }
}

// rows: of all experts
extern "C" void launch_moe_pack(const void* w, const void* scale,
                                const void* offset, void* out, int rows, int K,
                                int bits, int gs, hipStream_t stream) {
  const dim3 grid((unsigned)(rows / 16 * (K / MR_UNIT))), block(WAVE);
  const int words = moe_pack_words(bits, gs);
  if (bits == 4) {
    moe_pack_kernel<4><<<grid, block, 0, stream>>>(
        (const unsigned*)w, (const unsigned short*)scale,
        (const unsigned short*)offset, (unsigned*)out, K, gs, words);
  } else {
    moe_pack_kernel<8><<<grid, block, 0, stream>>>(
        (const unsigned*)w, (const unsigned short*)scale,
        (const unsigned short*)offset, (unsigned*)out, K, gs, words);
  }
}

// 2^32 / n, rounded up, for n above 1
static unsigned reciprocal(unsigned n) {
  return (unsigned)(((1ull << 32) + n - 1) / n);
}

template <int BITS, int GS, bool UP, bool FEW>
static void moe_rows_run(MoeRowsArgs a, hipStream_t stream) {
  // Two blocks a CU, all at work at once (64 tokens, 64 experts, 4 bits: 89 us; 116 with
  // one, 103 with four), or a tile each where there are fewer.  One where a CU holds one:
  // a block without a tile, of which there may be many, is then in the way of one that has
  // some (6 tokens of 16 experts of 1024 x 3072 in bf16, first product: 384 blocks 30.1
  // us, 256 18.8).
  auto go = [&](auto kernel, int resident) {
    const int tiles = a.O / 16 * min(a.experts, a.pairs);
    const int room = max(resident - a.dense, resident / 2);
    const unsigned blocks = min(room, tiles);
    a.by_blocks = reciprocal(blocks);
    a.by_rows = reciprocal(a.O / 16);
    kernel<<<dim3(a.dense + blocks), dim3(MR_BLOCK), 0, stream>>>(a);
  };
#define MR_GO(U) go(&moe_rows_kernel<BITS, GS, U, UP, FEW>, two_a_cu<BITS, U, UP>() ? 512 : 256)
  const int upw = (a.K / MR_UNIT + MR_WAVES - 1) / MR_WAVES;
  if (upw <= 1) {
    MR_GO(1);
  } else if (upw <= 2) {
    MR_GO(2);
  } else if (upw <= 3) {
    MR_GO(3);
  } else if constexpr (BITS < 16) {
    if (upw <= 4) MR_GO(4);
    else MR_GO(5);
  }
#undef MR_GO
}

template <int BITS, int GS, bool UP>
static void moe_rows_go(const MoeRowsArgs& a, hipStream_t stream) {
  if (a.pairs <= WAVE) moe_rows_run<BITS, GS, UP, true>(a, stream);
  else moe_rows_run<BITS, GS, UP, false>(a, stream);
}

// the longest contraction
extern "C" int moe_rows_longest(int bits) {
  return MR_UNIT * MR_WAVES * (bits < 16 ? 5 : 3);
}

template <bool UP>
static void moe_rows_pick(const MoeRowsArgs& a, int bits, int gs,
                          hipStream_t stream) {
  if (bits == 16) {
    moe_rows_go<16, MR_UNIT, UP>(a, stream);
  } else if (bits == 4) {
    if (gs == 32) moe_rows_go<4, 32, UP>(a, stream);
    else if (gs == 64) moe_rows_go<4, 64, UP>(a, stream);
    else moe_rows_go<4, 128, UP>(a, stream);
  } else {
    if (gs == 32) moe_rows_go<8, 32, UP>(a, stream);
    else if (gs == 64) moe_rows_go<8, 64, UP>(a, stream);
    else moe_rows_go<8, 128, UP>(a, stream);
  }
}

// K: whole units, as many as registers hold (moe_rows_longest); O: whole tiles of
// 16 rows; at most MR_PAIRS pairs.
extern "C" void launch_moe_rows(const MoeRowsArgs* a, int bits, int gs,
                                bool up, hipStream_t stream) {
  if (up) moe_rows_pick<true>(*a, bits, gs, stream);
  else moe_rows_pick<false>(*a, bits, gs, stream);
}

// -- router -----------------------------------------------------------------

// A block per token.  The router's product runs on the matrix cores with the
// token in every column: a wave has 16 experts and a quarter of the contraction,
// and asks for its weights (64 x H, out of L2) before the norm, which waits for
// rows and sums meanwhile: all of this is latency.
__global__ __launch_bounds__(1024) void moe_route_kernel(const MoeRouteArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __bf16* row = reinterpret_cast<__bf16*>(smem);     // [H]
  __shared__ float scratch[16];
  __shared__ float part[4][64];
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lg = lane >> 4, eg = wid & 3, quarter = wid >> 2;
  const long t = blockIdx.x;

  // This thread's columns of the row, up to 8192 of which rows have; they are
  // asked for ahead of the router's weights, as loads come back in order.
  const int col = threadIdx.x * 8;
  bf16x8_t v, r, n;
  if (col < a.H) {
    v = *reinterpret_cast<const bf16x8_t*>(a.x + t * a.H + col);
    if (a.residual)
      r = *reinterpret_cast<const bf16x8_t*>(a.residual + t * a.H + col);
    n = *reinterpret_cast<const bf16x8_t*>(a.norm + col);
  }
  const int steps = a.H / 128;  // of 32, of this quarter
  const bool works = eg * 16 < a.E;
  const __bf16* g = a.gate + (long)min(eg * 16 + (lane & 15), a.E - 1) * a.H +
                    quarter * steps * 32 + lg * 8;
  bf16x8_t w[16];
  if (works) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      w[i] = *reinterpret_cast<const bf16x8_t*>(g + min(i, steps - 1) * 32);
  }

  float ss = 0.0f;
  if (col < a.H) {
    if (a.residual) {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = (__bf16)((float)v[j] + (float)r[j]);
      *reinterpret_cast<bf16x8_t*>(a.h + t * a.H + col) = v;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) ss = fmaf((float)v[j], (float)v[j], ss);
  }
  ss = block_sum<1024>(ss, scratch);
  const float f = rsqrtf(ss / a.H + a.eps);
  if (col < a.H) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[j] = (__bf16)((float)v[j] * f * ((float)n[j] + a.offset));
    *reinterpret_cast<bf16x8_t*>(row + col) = v;
    *reinterpret_cast<bf16x8_t*>(a.y + t * a.H + col) = v;
  }
  __syncthreads();

  if (works) {
    const __bf16* x = row + quarter * steps * 32 + lg * 8;
    f32x4 acc[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
    for (int s = 0; s < steps; s += 16) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (s + i < steps)
          acc[i & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              w[i], *reinterpret_cast<const bf16x8_t*>(x + (s + i) * 32),
              acc[i & 1], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (s + 16 + i < steps)
          w[i] = *reinterpret_cast<const bf16x8_t*>(g + (s + 16 + i) * 32);
    }
    if ((lane & 15) == 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        part[quarter][eg * 16 + lg * 4 + r] = acc[0][r] + acc[1][r];
    }
  }
  __syncthreads();
  if (wid != 0) return;
  const float z = lane < a.E ? (part[0][lane] + part[1][lane]) +
                                   (part[2][lane] + part[3][lane])
                             : -INFINITY;
  int place;
  float weight;
  if (chosen_expert(z, lane, a.E, a.top, a.normalize, a.scaling, place, weight)) {
    a.choice[t * a.top + place] = lane;
    a.weight[t * a.top + place] = weight;
  }
}

// The same with a block for every 16 experts of a token: a CU reads about 30 bytes a
// nanosecond, 8.5 us for all weights of 64 experts of 2048.  The last block of a token
// has all logits, which pass the XCDs' L2s by accesses of the device's scope, and chooses.
// One token: 13.0 -> 8.7 us, 64: 13.2 -> 9.1.
__global__ __launch_bounds__(256) void moe_route_parts_kernel(const MoeRouteArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __bf16* row = reinterpret_cast<__bf16*>(smem);  // [H]
  __shared__ float scratch[4];
  __shared__ float part[4][16];
  const int lane = threadIdx.x & (WAVE - 1);
  const int quarter = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lg = lane >> 4, first = blockIdx.y * 16;
  const long t = blockIdx.x;

  auto load = [](const __bf16* p) { return *reinterpret_cast<const bf16x8_t*>(p); };
  bf16x8_t v[4], r[4], n[4];  // up to 8192 columns
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int col = (i * 256 + threadIdx.x) * 8;
    if (col >= a.H) continue;
    v[i] = load(a.x + t * a.H + col);
    if (a.residual) r[i] = load(a.residual + t * a.H + col);
    n[i] = load(a.norm + col);
  }
  const int steps = a.H / 128;  // of 32, of this quarter
  const __bf16* g = a.gate + (long)min(first + (lane & 15), a.E - 1) * a.H +
                    quarter * steps * 32 + lg * 8;
  bf16x8_t w[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) w[i] = load(g + min(i, steps - 1) * 32);

  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int col = (i * 256 + threadIdx.x) * 8;
    if (col >= a.H) continue;
    if (a.residual) {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[i][j] = (__bf16)((float)v[i][j] + (float)r[i][j]);
      if (blockIdx.y == 0) *reinterpret_cast<bf16x8_t*>(a.h + t * a.H + col) = v[i];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) ss = fmaf((float)v[i][j], (float)v[i][j], ss);
  }
  ss = block_sum<256>(ss, scratch);
  const float f = rsqrtf(ss / a.H + a.eps);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int col = (i * 256 + threadIdx.x) * 8;
    if (col >= a.H) continue;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[i][j] = (__bf16)((float)v[i][j] * f * ((float)n[i][j] + a.offset));
    *reinterpret_cast<bf16x8_t*>(row + col) = v[i];
    if (blockIdx.y == 0) *reinterpret_cast<bf16x8_t*>(a.y + t * a.H + col) = v[i];
  }
  __syncthreads();

  const __bf16* x = row + quarter * steps * 32 + lg * 8;
  f32x4 acc[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
  for (int s = 0; s < steps; s += 16) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (s + i < steps)
        acc[i & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i], load(x + (s + i) * 32),
                                                             acc[i & 1], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (s + 16 + i < steps) w[i] = load(g + (s + 16 + i) * 32);
  }
  if ((lane & 15) == 0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) part[quarter][lg * 4 + j] = acc[0][j] + acc[1][j];
  }
  __syncthreads();
  if (quarter != 0) return;
  float* logits = a.logits + t * 64;
  if (lane < 16)
    __hip_atomic_store(logits + first + lane,
                       (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  unsigned before = 0;
  if (lane == 0)
    before = __hip_atomic_fetch_add(a.tickets + t, 1u, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT);
  if (__builtin_amdgcn_readfirstlane(before) + 1 != gridDim.y) return;
  asm volatile("" ::: "memory");
  const float z = lane < a.E ? __hip_atomic_load(logits + lane, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT)
                             : -INFINITY;
  int place;
  float weight;
  if (chosen_expert(z, lane, a.E, a.top, a.normalize, a.scaling, place, weight)) {
    a.choice[t * a.top + place] = lane;
    a.weight[t * a.top + place] = weight;
  }
}

extern "C" void launch_moe_route(const MoeRouteArgs* a, int N,
                                 hipStream_t stream) {
  const size_t smem = (size_t)a->H * 2;
  if (a->tickets) {
    moe_route_parts_kernel<<<dim3((unsigned)N, (unsigned)((a->E + 15) / 16)), dim3(256),
                             smem, stream>>>(*a);
  } else {
    moe_route_kernel<<<dim3((unsigned)N), dim3(1024), smem, stream>>>(*a);
  }
}

// -- sum --------------------------------------------------------------------

__global__ __launch_bounds__(256) void moe_combine_kernel(
    const float* __restrict__ rows, const __bf16* __restrict__ h,
    const __bf16* __restrict__ shared, __bf16* __restrict__ out, int H, int top) {
  const long t = blockIdx.x;
  for (int i = (blockIdx.y * 256 + threadIdx.x) * 4; i < H;
       i += 256 * 4 * gridDim.y) {
    f32x4 v = {0, 0, 0, 0};
#pragma unroll 8
    for (int k = 0; k < top; ++k) {
      const f32x4 r =
          *reinterpret_cast<const f32x4*>(rows + (t * top + k) * H + i);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] += r[j];
    }
    bf16x4_t o;
    if (shared) {
      const bf16x4_t s = *reinterpret_cast<const bf16x4_t*>(shared + t * H + i);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] += (float)s[j];
    }
    if (h) {
      const bf16x4_t r = *reinterpret_cast<const bf16x4_t*>(h + t * H + i);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] += (float)r[j];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = (__bf16)v[j];
    *reinterpret_cast<bf16x4_t*>(out + t * H + i) = o;
  }
}

extern "C" void launch_moe_combine(const float* rows, const void* h,
                                   const void* shared, void* out, int N, int H,
                                   int top, hipStream_t stream) {
  const unsigned parts = (unsigned)((H + 1023) / 1024);
  moe_combine_kernel<<<dim3((unsigned)N, parts), dim3(256), 0, stream>>>(
      rows, (const __bf16*)h, (const __bf16*)shared, (__bf16*)out, H, top);
}
