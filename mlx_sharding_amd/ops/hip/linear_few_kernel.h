// What the kernels of products of few rows (linear_few.hip, linear_own.hip) share:
// arguments, where blocks begin, what happens to a tile's sums.
#pragma once

#include "hip_common.h"
#include "warm.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Two lines of 64 bytes, which a block asks for at once: numbers of a third line, or of the
// second when the first had come, took every launch 0.4 us.
struct LinearFewArgs {
  const __bf16 *x, *w, *bias, *res, *norm;
  __bf16* y;
  short M;
  // parts > 1: blocks share a tile's contraction, `share` stages each.  part [tiles of y,
  // parts, tiles of x, WAVE, 4], count: one number per tile of y and x, zero before.
  // (linear_own.hip: the unit, and the chunks or stages of the whole contraction)
  unsigned char parts;
  unsigned char fours;     // bias and residual are read by fours
  int O, K;                // O: columns of y
  int share;
  long ldx, ldw, ldr, ldy;
  union {
    struct { float eps, offset; };  // norm weights are norm + offset
    float* part;                    // without a norm
  };
  unsigned turn;           // 2^32 / chunks of a share, rounded up, for first_of
  int n_zero;              // numbers at zero that this launch clears for a later one
  unsigned *count, *zero;
};
static_assert(sizeof(LinearFewArgs) == 128, "two lines");

// all of a, now
__device__ __forceinline__ void arrive(const LinearFewArgs& a) {
  asm volatile("" ::"s"(a.x), "s"(a.w), "s"(a.bias), "s"(a.res), "s"(a.norm), "s"(a.O),
               "s"(a.K), "s"(a.share), "s"(a.ldx), "s"(a.ldw), "s"(a.turn), "s"(a.zero));
}

// Where a block begins in the n chunks of a contraction; it goes round from there.
// Where rows of W lie in step (in_step), blocks at one column ask few of the memory's
// channels: 16384 rows of 2048, 12 of x, 16.4 us from column 0 on, 14.1 so (the blocks of an
// XCD, which are every eighth, three chunks apart; one apart 14.2, seven 14.5); 28672 of 4096
// with norm and unit 45.6, 43.5; 6144 of 4096 14.7, 13.2; 14080 of 5504, 8 of x, 39.3, 32.5;
// 64 of x, four tiles, rows of 4096 .87 of the time.  Others need none, and going round costs
// them up to 10% (turn 0: 8 of x, 16064 units of 5376 64.0 us from column 0 on, 70.2 else; one
// of x, 7008 rows of 16192 42.6, 46.8).  `turn` divides by the chunks of a whole share: the
// last may have less.
__device__ __forceinline__ int first_of(const LinearFewArgs& a, int whole, int n,
                                        unsigned block) {
  return first_chunk(a.turn, whole, n, block);
}

// The sums of a tile that blocks share: leaves this one's, and true in the one that
// comes last, which then has all, added in the blocks' order.  Sums pass the L2s, which
// XCDs have of their own, by accesses of the device's scope.
__device__ __forceinline__ bool sums_of_all(const LinearFewArgs& a, long tile,
                                            int lane, f32x4& v) {
  typedef unsigned long long u64;
  typedef u64 u64x2 __attribute__((ext_vector_type(2)));
  u64* to = reinterpret_cast<u64*>(a.part) + (tile * a.parts * WAVE + lane) * 2;
  const u64x2 own = __builtin_bit_cast(u64x2, v);
#pragma unroll
  for (int i = 0; i < 2; ++i)
    __hip_atomic_store(to + blockIdx.y * (WAVE * 2) + i, own[i], __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  unsigned before = 0;
  if (lane == 0)
    before = __hip_atomic_fetch_add(a.count + tile, 1u, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT);
  before = __builtin_amdgcn_readfirstlane(before);
  if (before + 1 != a.parts) return false;
  asm volatile("" ::: "memory");
  v = f32x4{0, 0, 0, 0};
#pragma unroll 4
  for (unsigned s = 0; s < a.parts; ++s) {
    u64x2 p;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      p[i] = __hip_atomic_load(to + s * (WAVE * 2) + i, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    const f32x4 f = __builtin_bit_cast(f32x4, p);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] += f[j];
  }
  return true;
}

// LF_CLAMPED: g = min(gate, eps), u = up within eps, g sigmoid(offset g) (u + 1), on the kernels
// of linear_own.hip, without a norm or a residual; of the first n_zero columns, bias is added to
// the gate and res, a vector like it, to the up projection
enum { LF_PLAIN = 0, LF_SILU = 1, LF_GELU = 2, LF_CLAMPED = 3 };

typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

// What is added to four columns of y, if it may be read by fours.  Asked for before the
// contraction: behind it, the residual's were four reads one after the other (us without
// and with a residual; one of x, 2048 rows of 2048 5.4 and 5.6, so 5.1 both; 12 of x, 4096
// of 4096 9.4 and 9.9, so 9.2 both; 64 of x 13.8 and 14.4, so 13.5 and 13.9).
template <int ACT>
struct Ends {
  bf16x4_t res, bias[ACT ? 2 : 1];

  __device__ __forceinline__ void read(const LinearFewArgs& a, int row, int col) {
    col = min(col, a.O - 4);
    if (a.res)
      res = *reinterpret_cast<const bf16x4_t*>(a.res + min(row, a.M - 1) * a.ldr + col);
    if (a.bias) {
#pragma unroll
      for (int h = 0; h < (ACT ? 2 : 1); ++h)
        bias[h] = *reinterpret_cast<const bf16x4_t*>(a.bias + h * a.O + col);
    }
  }
};

// sums of four columns of y from `col` on, and of an up projection's, to memory
template <int ACT>
__device__ __forceinline__ void finish_columns(const LinearFewArgs& a, int row, int col,
                                               const f32x4* v, const Ends<ACT>& e) {
  float o[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int at = min(col + j, a.O - 1);
    float f = v[0][j];
    if (ACT) {
      float up = v[1][j];
      if (a.bias) {
        f += (float)(a.fours ? e.bias[0][j] : a.bias[at]);
        up += (float)(a.fours ? e.bias[ACT ? 1 : 0][j] : a.bias[a.O + at]);
      }
      if (ACT == LF_SILU) {
        f = f / (1.0f + __expf(-f)) * up;
      } else {
        const float z = 0.7978845608028654f * (f + 0.044715f * f * f * f);
        f = 0.5f * f * (1.0f + tanhf(z)) * up;
      }
    } else if (a.bias) {
      f += (float)(a.fours ? e.bias[0][j] : a.bias[at]);
    }
    if (a.res) f += (float)(a.fours ? e.res[j] : a.res[(long)row * a.ldr + at]);
    o[j] = f;
  }
  __bf16* y = a.y + (long)row * a.ldy + col;
  if (col + 3 < a.O && a.ldy % 4 == 0) {
    *reinterpret_cast<bf16x4_t*>(y) =
        bf16x4_t{(__bf16)o[0], (__bf16)o[1], (__bf16)o[2], (__bf16)o[3]};
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (col + j < a.O) y[j] = (__bf16)o[j];
  }
}

// Whether rows that lie ld apart meet the same few of the memory's channels: up to five of
// them are a multiple of 16 KB, or miss it by less than a channel's 256 bytes.
static bool in_step(long ld) {
  for (int n = 1; n <= 5; ++n) {
    const int off = (int)(n * ld * 2 % 16384);
    if (min(off, 16384 - off) <= 256) return true;
  }
  return false;
}

// Products of whole contractions on the kernels of linear_own.hip, or false where they are
// linear_few.hip's.
bool linear_own_go(LinearFewArgs a, int act, hipStream_t stream);
// A contraction that `split` blocks share, for up to 16 rows of x.
void linear_own_shared(LinearFewArgs a, int split, hipStream_t stream);
