// y = x W^T for few rows of x (decoding, short prompts): what lies between two such products of
// a layer goes with them.
//
//   before:  RMS norm of x's rows with a weight per column
//   behind:  bias, residual rows, or the gated unit act(gate) * up of two halves
//            of W's rows
//
// Bound by reading W once; a short kernel also by launch and latency, so each
// operation taken along saves its launch (2 to 4 us within a captured step).
// W and x go to LDS in whole lines and from there to operands of 16x16x32 products; the waves of
// a block take the contraction by turns and add up through LDS.  x comes from L2, once per
// block.  The norm's factor is applied to the sums: x times the weight is rounded to bf16, as
// the normed row was.
// Whole contractions are linear_own.hip's but for one size of block; here are that and
// contractions that blocks share.
// Measured with weights out of memory (sets of 1.5 GB and more by turns), beside the
// library's product (us; M x K x O): 1 x 2048 x 2048: 4.0, 11.0; 1 x 4096 x 4096: 8.3, 15.5;
// 64 x 2048 x 2048: 5.6, 11.7; 64 x 4096 x 4096: 13.0, 15.1; 64 x 2048 x 11264: 15.4, 16.0;
// 64 x 4096 x 28672: 45, 53; 64 x 14336 x 4096, shared: 29, 39.  With norm and unit, 1 x 4096 x
// 28672: 40 (5.9 TB/s), beside 72 for three kernels.

#include "linear_few_kernel.h"

// Waves meet at stages of KS steps of 32 columns, in a ring; a wave takes one of the steps, for
// all rows of W and of x or for half of x's.  W to registers by rows of 64 bytes: 10.6 us for
// 64 x 2048 x 2048, 70 for 64 x 4096 x 28672.
#define LS_WAVES 8

// What blocks have of a contraction: all of it, from the first column on or, where the memory
// asks for it, from a column of their own (first_of), or a share.
enum { LS_WHOLE = 0, LS_TURNED = 1, LS_SHARED = 2 };

// RT, TT: tiles of 16 rows of W and of x
template <int RT, int TT, int ACT, int WAY>
__global__ __launch_bounds__(LS_WAVES * WAVE) void linear_some_kernel(
    const LinearFewArgs a) {
  constexpr int KS = 4, YT = ACT ? RT / 2 : RT;
  constexpr int PARTS = (RT + TT) * KS / LS_WAVES;  // loads to LDS, wave and stage
  constexpr int STAGE = (RT + TT) * KS * 1024;
  constexpr int RING = 4 * STAGE > 140 * 1024 ? 3 : 4;
  // loads of a wave that may be under way when it comes to a stage
  constexpr int BEHIND = (RING - 2) * PARTS;
  constexpr int TW = TT * KS / LS_WAVES;            // tiles of x of a wave
  constexpr int RP = KS * 4;                        // pieces of 16 bytes of a row
  extern __shared__ __attribute__((aligned(16))) char smem[];

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
  };
  f32x4 acc[RT][TW];
#pragma unroll
  for (int i = 0; i < TW; ++i)
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[r][i] = f32x4{0, 0, 0, 0};
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
    for (int i = 0; i < TW; ++i)
#pragma unroll
      for (int r = 0; r < RT; ++r)
        acc[r][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[r], v[i], acc[r][i],
                                                            0, 0, 0);
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
    if (WAY == LS_SHARED &&
        !sums_of_all(a, ((long)blockIdx.x * YT + r) * TT + i, lane, v[0]))
      continue;
    if (i * 16 + l16 < a.M)
      finish_columns<ACT>(a, i * 16 + l16, row0 + r * 16 + lg * 4, v, ends[q]);
  }
}

// Blocks that share a tile's contraction, as many as have something of it.
static dim3 shared_grid(LinearFewArgs& a, int cols, int steps, int split) {
  a.share = (steps + split - 1) / split;
  const int parts = (steps + a.share - 1) / a.share;
  a.parts = (unsigned char)parts;
  a.turn = a.share > 1 && in_step(a.ldw)
               ? (unsigned)(((1ull << 32) + a.share - 1) / a.share) : 0;
  return dim3((unsigned)((a.O + cols - 1) / cols), (unsigned)parts);
}

template <int RT, int TT, int ACT>
static void linear_some_go(LinearFewArgs a, int split, hipStream_t stream) {
  constexpr int KS = 4, cols = 16 * (ACT ? RT / 2 : RT);
  constexpr int stage = (RT + TT) * KS * 1024;
  constexpr int ring = (4 * stage > 140 * 1024 ? 3 : 4) * stage;
  constexpr int smem = ring > KS * RT * TT * 1024 ? ring : KS * RT * TT * 1024;
  const dim3 grid = shared_grid(a, cols, (a.K + KS * 32 - 1) / (KS * 32), split);
  auto go = [&](auto kernel) {
    if (smem > 56 * 1024)  // above the default limit
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    kernel<<<grid, dim3(LS_WAVES * WAVE), smem, stream>>>(a);
  };
  if constexpr (!ACT) {
    if (RT == 2 || a.parts > 1) return go(&linear_some_kernel<RT, TT, ACT, LS_SHARED>);
  }
  if constexpr (RT == 4) {
    if (a.turn) go(&linear_some_kernel<RT, TT, ACT, LS_TURNED>);
    else go(&linear_some_kernel<RT, TT, ACT, LS_WHOLE>);
  }
}

template <int TT>
static void linear_some(const LinearFewArgs& a, int act, int split, hipStream_t stream) {
  if (split > 1 && a.O <= 2048) linear_some_go<2, TT, LF_PLAIN>(a, split, stream);
  else if (act == LF_SILU) linear_some_go<4, TT, LF_SILU>(a, 1, stream);
  else if (act == LF_GELU) linear_some_go<4, TT, LF_GELU>(a, 1, stream);
  else linear_some_go<4, TT, LF_PLAIN>(a, split, stream);
}

// Blocks that share a tile's contraction where the caller has room for their sums, as many
// as come in one round: x is read once per block, four times W with 16 rows of W and 64 of
// x, so that long rows have blocks of more rows and a part of the columns each, and up to
// 2048 rows of W leave CUs idle without.  Blocks have two tiles up to there and four above.
// Shared and whole (linear_own.hip; us): 64 of x, 1536 rows of 2816 7.4, 5.8, 1616 of 4288
// 10.2, 9.5, 1504 of 5632 10.9, 11.3, 2048 of 8704 16.7, 19.1, 3072 of 9216 22.6, 24.8; 29 of
// x, 2048 of 9216 12.7, 15.3.  In two rounds it loses (64 of x, 2816 rows of 4096 17.4, 19.9).
// Up to 16 of x go the waves' own rings, 16 rows of W a block, by two blocks or, up to 1024
// rows, by four: time over that of whole ones up to 1024 rows of 4096 to 5632 1.04, to 8192
// .80, to 12288 .65, to 2048 rows of 5632 to 8192 .87, to 12288 .80; more rows 1.0 to 1.2.
static int few_split(int M, int O, int K, int act, bool norm) {
  if (act || norm) return 1;
  if (M <= 16) return O <= 2048 && K >= 5632 ? (O <= 1024 ? 4 : 2) : 1;
  if (O <= 2048) return K >= (M > 32 ? 5632 : 7168) ? 4 : 1;
  return K >= 8192 && O <= 4096 ? 4 : 1;
}

// Room for a shared contraction: `numbers` to be cleared before, and sums behind them.
extern "C" long linear_few_room(int M, int O, int K, int* numbers) {
  const int split = few_split(M, O, K, 0, false);
  const int tiles = (O + 63) / 64 * 4 * ((M + 31) / 32 * 2);
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
  if (norm || act == LF_CLAMPED) a.eps = eps, a.offset = offset;
  else a.part = part;
  a.count = count, a.zero = zero, a.n_zero = n_zero;
  a.fours = (bias || res) && O % 4 == 0 && (long)bias % 8 == 0 && (long)res % 8 == 0 &&
            (!res || ldr % 4 == 0);
  const int split = count ? few_split(M, O, K, act, norm != nullptr) : 1;
  if (split == 1 && linear_own_go(a, act, stream)) return;
  if (M <= 16) linear_own_shared(a, split, stream);
  else if (M <= 32) linear_some<2>(a, act, split, stream);
  else linear_some<4>(a, act, split, stream);
}
