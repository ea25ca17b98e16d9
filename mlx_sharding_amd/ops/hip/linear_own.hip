// y = x W^T for up to 64 rows of x, whole contractions (what goes along: linear_few.hip).
//
// A CU reads rows through LDS at 100 bytes a nanosecond and more as long as a load takes
// whole lines (128 bytes of 8 rows; 64 bytes of 16 rows, as operands straight to registers
// are: 35), so that products of up to 30 MB are not bound by what a block reads of x, but by
// the chain of its stages: the waves of linear_some_kernel meet at each one, 0.6 us of which
// are 0.35 of reads from LDS and products and, with a norm, 0.85 (64 rows of 2048 into 3648).
// Two kernels without it:
//
//   linear_own_kernel   each wave has a ring of its own in LDS and takes chunks of 64 columns
//                       by turns, so that no wave waits for another before the sums; for up
//                       to four tiles of W's rows, and five and seven of up to 16 rows of x
//   linear_ring_kernel  five to eight tiles, which is more than such rings have room for:
//                       waves meet, half of them load W, half x, in rings of lengths that
//                       suit each
//
// Tiles are as many as make blocks one round of the chip where two and four would leave a second
// one half empty, and rows of x may be split between blocks that lie eight apart, on one XCD,
// whose L2 then has W's rows for both.
#include "linear_own_kernel.h"

namespace {

template <int RT, int TT, int SL, int GATED, bool NORM, bool SHARED, bool PAIRS = false>
__global__ __launch_bounds__(OWN_WAVES * WAVE) void linear_own_kernel(const LinearFewArgs a) {
  own_block<RT, TT, SL, GATED, NORM, SHARED, PAIRS>(a, blockIdx.x);
}

// RT, TT as above (one group of x's rows); RW, RX: stages of 128 columns of W and of x in
// LDS, a row of the norm's weights behind x's.
template <int RT, int TT, int RW, int RX, int GATED, bool NORM>
__global__ __launch_bounds__(OWN_WAVES * WAVE) void linear_ring_kernel(const LinearFewArgs a) {
  constexpr int KS = 4, TW = TT * KS / OWN_WAVES;  // steps of a stage, tiles of x of a wave
  constexpr int COLS = (GATED ? 8 : 16) * RT;
  constexpr int SW = RT * 4096, SX = TT * 4096 + (NORM ? 1024 : 0), XS = RW * SW;
  constexpr int MOST = RT > TT ? RT : TT;  // loads of a wave and stage: RT or TT
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ float squares[NORM ? OWN_WAVES : 1][TW][WAVE];

  arrive(a);
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int l16 = lane & 15, lg = lane >> 4;
  const int step = wid % KS, tile0 = wid / KS * TW, part = wid & 3;
  const BlockPlace at = place_of(a, 16 * TT, blockIdx.x);
  const int x0 = at.x0, col0 = at.bx * COLS;
  if (col0 >= a.O) return;
  const bool loads_w = wid < 4;

  // a load is 4 rows of 256 bytes, pieces swapped by the row
  const char* from[MOST];
  int col[MOST];
#pragma unroll
  for (int i = 0; i < MOST; ++i) {
    const int row = (i * 4 + part) * 4 + (lane >> 4);
    col[i] = ((lane & 15) ^ (row & 15)) * 8;
    from[i] = (const char*)(loads_w ? row_of<GATED>(a, col0, row)
                                    : a.x + (long)min(x0 + row, a.M - 1) * a.ldx);
  }
  constexpr int W = KS * 32;  // columns of a stage
  const int stages = (a.K + W - 1) / W;
  const int first = first_of(a, a.share, stages, at.bx);
  auto column = [&](int t) {
    const int c = t + first;
    return (c >= stages ? c - stages : c) * W;
  };
  const unsigned lds = lds_at(smem);
  auto issue_w = [&](int t, int slot) {
    const int k0 = column(t);
#pragma unroll
    for (int i = 0; i < RT; ++i)
      to_lds(from[i] + (unsigned)min(k0 + col[i], a.K - 8) * 2,
             lds + slot * SW + (i * 4 + part) * 1024);
  };
  auto issue_x = [&](int t, int slot) {
    const int k0 = column(t);
#pragma unroll
    for (int i = 0; i < TT; ++i)
      to_lds(from[i] + (unsigned)min(k0 + col[i], a.K - 8) * 2,
             lds + XS + slot * SX + (i * 4 + part) * 1024);
    if (NORM)  // the same from each of the four waves
      to_lds((const char*)(a.norm + min(k0 + (lane & 15) * 8, a.K - 8)),
             lds + XS + slot * SX + TT * 4096);
  };
  f32x4 acc[RT][TW];
  float sq[TW];
#pragma unroll
  for (int i = 0; i < TW; ++i) {
    sq[i] = 0.0f;
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[r][i] = f32x4{0, 0, 0, 0};
  }
  const int piece = l16 * 256 + ((step * 4 + lg) ^ l16) * 16;
  if (loads_w) {
#pragma unroll
    for (int t = 0; t < RW - 1; ++t)
      if (t < stages) issue_w(t, t);
  } else {
#pragma unroll
    for (int t = 0; t < RX - 1; ++t)
      if (t < stages) issue_x(t, t);
  }
  constexpr int TILES = (RT * TT + OWN_WAVES - 1) / OWN_WAVES;  // of y, of a wave
  Ends<0> ends[TILES];
  if (!GATED && a.fours) {
#pragma unroll
    for (int q = 0; q < TILES; ++q) {
      const int n = min(wid + q * OWN_WAVES, RT * TT - 1);
      ends[q].read(a, x0 + n % TT * 16 + l16, col0 + n / TT * 16 + lg * 4);
    }
  }
  int sw = 0, sx = 0;
  for (int t = 0; t < stages; ++t) {
    if (loads_w) wait_chunks<RW - 2, RT>(stages - 1 - t);
    else wait_chunks<RX - 2, TT + (NORM ? 1 : 0)>(stages - 1 - t);
    meet();
    // into the place of the stage before, which all have read
    if (loads_w) {
      if (t + RW - 1 < stages) issue_w(t + RW - 1, sw ? sw - 1 : RW - 1);
    } else if (t + RX - 1 < stages) {
      issue_x(t + RX - 1, sx ? sx - 1 : RX - 1);
    }
    if (column(t) + step * 32 < a.K) {
      const char* wb = smem + sw * SW + piece;
      const char* xb = smem + XS + sx * SX + piece;
      bf16x8_t w[RT], v[TW], g;
#pragma unroll
      for (int i = 0; i < TW; ++i)
        v[i] = *reinterpret_cast<const bf16x8_t*>(xb + (tile0 + i) * 4096);
      if (NORM)
        g = *reinterpret_cast<const bf16x8_t*>(smem + XS + sx * SX + TT * 4096 +
                                               (step * 4 + lg) * 16);
#pragma unroll
      for (int r = 0; r < RT; ++r) w[r] = *reinterpret_cast<const bf16x8_t*>(wb + r * 4096);
#pragma unroll
      for (int i = 0; i < TW; ++i) {
        const bf16x8_t x = NORM ? times(v[i], g, a.offset, sq[i]) : v[i];
#pragma unroll
        for (int r = 0; r < RT; ++r)
          acc[r][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[r], x, acc[r][i], 0, 0, 0);
      }
    }
    if (++sw == RW) sw = 0;
    if (++sx == RX) sx = 0;
  }
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
    for (int i = threadIdx.x; i < a.n_zero; i += OWN_WAVES * WAVE) a.zero[i] = 0;
#pragma unroll
  for (int q = 0; q < TILES; ++q) {
    const int n = wid + q * OWN_WAVES;
    if (n >= RT * TT) break;
    const f32x4 v = sum_of<TT, KS, TW, NORM>(a, red, squares, RT * TT, n, lane);
    const int row = x0 + n % TT * 16 + l16;
    if (row < a.M)
      finish_tile<GATED>(a, row, col0 + n / TT * (GATED ? 8 : 16), lg, v, ends[q]);
  }
}

template <typename Kernel>
void launch(Kernel kernel, const LinearFewArgs& a, int blocks, int smem, hipStream_t stream) {
  if (smem > 48 * 1024)  // with the sums of squares above the default limit
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  kernel<<<blocks, OWN_WAVES * WAVE, smem, stream>>>(a);
}

template <int RT, int TT>
void own(LinearFewArgs a, int act, hipStream_t stream) {
  const int cols = (act ? 8 : 16) * RT, groups = (a.M + 16 * TT - 1) / (16 * TT);
  int blocks = (a.O + cols - 1) / cols;
  if (groups > 1) blocks = (blocks + 7) / 8 * 8 * groups;
  turned(a, act, 64);
  // Two chunks of a wave where blocks are small; a norm's instructions cover for one (64 rows
  // of 2048 into 3648: 8.8 us with one, 9.5 with two) but in long rows of few (1 to 16 rows
  // of 2048 to 4096 .98, of more than 6144 .90).
  constexpr int most = RT == 1 || (RT == 2 && TT == 2) ? 2 : 1;
  static_assert(own_room(RT, TT, most, 0, false) <= OWN_LDS, "room of the chunks that it has");
  auto go = [&](auto kernel, int slots) {
    launch(kernel, a, blocks, own_room(RT, TT, slots, a.K, a.norm != nullptr), stream);
  };
  if (a.norm) {
    if constexpr (RT == 1 && TT == 1) {
      if (a.K >= 2048 && own_room(RT, TT, most, a.K, true) <= OWN_LDS) {
        if (act) return go(&linear_own_kernel<RT, TT, most, true, true, false>, most);
        return go(&linear_own_kernel<RT, TT, most, false, true, false>, most);
      }
    }
    if (act) go(&linear_own_kernel<RT, TT, 1, true, true, false>, 1);
    else go(&linear_own_kernel<RT, TT, 1, false, true, false>, 1);
  } else {
    if (act == LF_CLAMPED) go(&linear_own_kernel<RT, TT, most, CLAMPED_ROWS, false, false>, most);
    else if (act) go(&linear_own_kernel<RT, TT, most, true, false, false>, most);
    else go(&linear_own_kernel<RT, TT, most, false, false, false>, most);
  }
}

template <int RT, int TT>
void ring(LinearFewArgs a, int act, hipStream_t stream) {
  constexpr int RW = TT == 2 ? (RT >= 7 ? 4 : 5) : (RT >= 7 ? 3 : 4), RX = TT == 2 && RT < 8 ? 4 : 3;
  const int cols = (act ? 8 : 16) * RT, groups = (a.M + 16 * TT - 1) / (16 * TT);
  int blocks = (a.O + cols - 1) / cols;
  if (groups > 1) blocks = (blocks + 7) / 8 * 8 * groups;
  turned(a, act, 128);
  auto go = [&](auto kernel) {
    const int rings = RW * RT * 4096 + RX * (TT * 4096 + (a.norm ? 1024 : 0));
    const int sums = RT * TT * 4096;
    launch(kernel, a, blocks, rings > sums ? rings : sums, stream);
  };
  if (a.norm) {
    if (act) go(&linear_ring_kernel<RT, TT, RW, RX, true, true>);
    else go(&linear_ring_kernel<RT, TT, RW, RX, false, true>);
  } else {
    if (act == LF_CLAMPED) go(&linear_ring_kernel<RT, TT, RW, RX, CLAMPED_ROWS, false>);
    else if (act) go(&linear_ring_kernel<RT, TT, RW, RX, true, false>);
    else go(&linear_ring_kernel<RT, TT, RW, RX, false, false>);
  }
}

// Tiles of W's rows and of x's.  What the busiest CU reads decides: its blocks, one after the
// other, times what a block reads, up to 16 rows of x as half a tile, as most of their loads
// find lines in L1, and where more than four tiles leave a CU one block, half a tile more.
// Where two read as much, fewer rows of x or tiles a block.  Over 650 random sizes of 17 to 64
// rows, with and without norm and unit, the kernels so chosen take .81 of the time of stages
// that waves meet at and .4% more than the fastest of 14 (us; 64 of x: units of 14336 of 4096
// with norm, seven tiles 60.2, 44.2; of 10944 of 2048, six 31.0, 22.3; 6144 of 4096 with norm,
// three of 32 rows of x 21.5, 17.0; 3648 of 2048 with norm, two of 32 11.4, 8.8; 2048 of 2048,
// one of 32 6.6, 5.6; 32 of x, one of 16 5.4, 4.8).  Over 350 of 1 to 16 rows they take .85 of
// the time of operands straight to registers and 1% more than the fastest (one of x: units of
// 14336 of 4096 with norm 43.3, 40.2, 6144 of 4096 13.2, 11.5, 2048 of 2048 4.7, 4.0; 5 of x,
// 3584 of 14336 22.6, 20.2; 12 of x, 12352 of 2048 12.3, 11.4; 16 of x, 4096 of 2048 7.3, 6.1).
// linear_some_kernel keeps what it does as well or better: four tiles for 17 and more rows of x
// in one block, without a norm (16176 rows of 2048 16.3, 17.3; units of 7408 of 1024 10.1,
// 11.3).
struct OwnTiles {
  int rt, tt;  // rt 0: linear_some_kernel's
};
OwnTiles own_tiles(int M, int O, int K, int act, bool norm) {
  const int tiles = (O + (act ? 7 : 15)) / (act ? 8 : 16);
  OwnTiles best{0, 0};
  long least = 0;
  auto offer = [&](int rt, int tt) {
    // Three and four tiles read in two rounds no more than these in one, and one of W beside
    // 64 rows of x no less than three beside 32: they would never be the first with the least.
    if ((tt == 1 && (rt == 6 || rt == 8)) || (rt == 1 && tt == 4)) return;
    if ((rt <= 4 || tt == 1) && own_room(rt, tt, 1, K, norm) > OWN_LDS) return;
    const long blocks = (long)(tiles + rt - 1) / rt * ((M + 16 * tt - 1) / (16 * tt));
    const int halves = M > 16 ? 2 * (rt + tt) : 2 * rt + 1 + (rt > 4);
    const long reads = (blocks + 255) / 256 * halves;
    if (!best.rt || reads < least || (reads == least && tt < best.tt))
      best = {rt, tt}, least = reads;
  };
  const int whole = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  for (int rt = 1; rt <= 8; ++rt) {
    offer(rt, whole);
    if (rt <= 4 && whole > 1) offer(rt, whole / 2);
  }
  if (!norm && best.rt == 4 && best.tt == whole && whole > 1) return {0, 0};
  return best;
}

// The same for 65 and more rows of x, where one round of blocks has them all: few tiles of 32
// rows or more of 64, whichever read less, and rt 0 where the kernels of more rows are the better
// ones.  Those wait for whole tiles of 128 rows of x and more, often on a part of the CUs; but
// what a block reads here grows with its tiles and the groups that read W, and from six tiles,
// from 384 rows or above contractions of 8192 they catch up (178 rows of 8192 into 7792, six
// tiles, 82.2 us here, 52.2; 299 of 14336 into 1984 50.8, 38.3).  Over 233 random sizes that are
// taken the time is .71 of theirs (us, before and now: 211 rows of 512 into 512 6.3, 3.0; 90 of
// 2048 into 1024 8.4, 4.6; 70 of 4096 into 3584 14.1, 10.3; 193 of 2048 into 4544 19.8, 13.1;
// units of 4096 of 74 of 5120 32.7, 28.9).  Contractions below 512 are not measured, and stay.
OwnTiles own_tiles_many(int M, int O, int K, int act) {
  const int tiles = (O + (act ? 7 : 15)) / (act ? 8 : 16);
  OwnTiles best{0, 0};
  if (M > 384 || K < 512 || K > 8192) return best;
  for (const int tt : {2, 4}) {
    const int groups = (M + 16 * tt - 1) / (16 * tt), most = tt == 2 ? 3 : M <= 128 ? 8 : 5;
    const int rt = (tiles + 256 / groups - 1) / (256 / groups);
    if (rt <= most && (!best.rt || rt + tt < best.rt + best.tt)) best = {rt, tt};
  }
  return best;
}

}  // namespace

// Whether the product of more than 64 rows, on its own, is one of these.
extern "C" int linear_own_many(long M, long O, long K, int act) {
  return M > 64 && M <= 384 && O >= 1 && O < 1 << 17 && K <= 8192 && K % 32 == 0 &&
         own_tiles_many((int)M, (int)O, (int)K, act).rt > 0;
}

// Blocks of a tile of up to 16 rows of x share its contraction.
void linear_own_shared(LinearFewArgs a, int split, hipStream_t stream) {
  turned(a, LF_PLAIN, 64);
  const int chunks = a.share;
  a.share = (chunks + split - 1) / split;
  a.parts = (unsigned char)((chunks + a.share - 1) / a.share);
  if (a.turn) a.turn = a.share > 1 ? (unsigned)(((1ull << 32) + a.share - 1) / a.share) : 0;
  const int smem = own_room(1, 1, 2, a.K, false);
  const auto kernel = &linear_own_kernel<1, 1, 2, false, false, true>;
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  kernel<<<dim3((unsigned)((a.O + 15) / 16), a.parts), OWN_WAVES * WAVE, smem, stream>>>(a);
}

bool linear_own_go(LinearFewArgs a, int act, hipStream_t stream) {
  OwnTiles t = a.M > 64 ? own_tiles_many(a.M, a.O, a.K, act)
                        : own_tiles(a.M, a.O, a.K, act, a.norm != nullptr);
  if (!t.rt && act == LF_CLAMPED) t = {4, a.M <= 32 ? 2 : 4};  // which has no other kernel
  switch (t.rt * 8 + t.tt) {
    case 1 * 8 + 1: own<1, 1>(a, act, stream); return true;
    case 2 * 8 + 1: own<2, 1>(a, act, stream); return true;
    case 3 * 8 + 1: own<3, 1>(a, act, stream); return true;
    case 4 * 8 + 1: own<4, 1>(a, act, stream); return true;
    case 5 * 8 + 1: own<5, 1>(a, act, stream); return true;
    case 7 * 8 + 1: own<7, 1>(a, act, stream); return true;
    case 1 * 8 + 2: own<1, 2>(a, act, stream); return true;
    case 2 * 8 + 2: own<2, 2>(a, act, stream); return true;
    case 3 * 8 + 2: own<3, 2>(a, act, stream); return true;
    case 4 * 8 + 2: own<4, 2>(a, act, stream); return true;
    case 2 * 8 + 4: own<2, 4>(a, act, stream); return true;
    case 3 * 8 + 4: own<3, 4>(a, act, stream); return true;
    case 4 * 8 + 4: own<4, 4>(a, act, stream); return true;
    case 5 * 8 + 2: ring<5, 2>(a, act, stream); return true;
    case 6 * 8 + 2: ring<6, 2>(a, act, stream); return true;
    case 7 * 8 + 2: ring<7, 2>(a, act, stream); return true;
    case 5 * 8 + 4: ring<5, 4>(a, act, stream); return true;
    case 6 * 8 + 4: ring<6, 4>(a, act, stream); return true;
    case 7 * 8 + 4: ring<7, 4>(a, act, stream); return true;
    case 8 * 8 + 2: ring<8, 2>(a, act, stream); return true;
    case 8 * 8 + 4: ring<8, 4>(a, act, stream); return true;
  }
  return false;
}

// Up to 28 MB in all: the L2s have 32 (a step of one sequence, 32 heads of 128 over 8, 4096 by
// 4096 behind them: 8 MB 402 us, 16 401, 24 to 40 398, none 406).  From 1.5 MB on: over 510 random
// layers of 1 to 16 sequences of 10 to 12000 keys, 317 of which this is for, a layer's time is
// .983 of that without it where the weights are 1.5 to 64 MB, 1.000 at 128 MB, 1.001 below 1.5 MB
// (1.005 at .25 MB), whose product is launch and latency alone.
extern "C" bool linear_own_warm(long M, long O, long K, long ld, const void* w, Warm* out) {
  if (M < 1 || M > 16 || O < 1 || O >= 1L << 24 || K < 512 || K >= 1L << 22 || K % 32 ||
      ld < K || ld >= 1L << 22 || O * K < 3L << 18)
    return false;
  LinearFewArgs a{};
  a.M = (short)M, a.O = (int)O, a.K = (int)K, a.ldw = ld;
  turned(a, LF_PLAIN, 64);
  const int rt = own_tiles(a.M, a.O, a.K, LF_PLAIN, false).rt;
  if (!rt) return false;
  const int blocks = (a.O + 16 * rt - 1) / (16 * rt);
  const long most = (28L << 20) / ((long)blocks * rt * 16 * 128);
  if (most < 1) return false;
  *out = Warm{(const char*)w, ld * 2, rt * 16, a.O, a.K, (int)min((long)a.share, most), blocks,
              a.turn};
  return true;
}
