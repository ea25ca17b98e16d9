// y = x W^T for few rows of x (decoding): what lies between two such products of
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
// Measured, beside the library's product (us; M x K x O): 1 x 2048 x 2048: 5.0,
// 11.0; 1 x 4096 x 4096: 8.4, 15.5; 1 x 4096 x 28672: 38 (6.2 TB/s), 62; 16 of
// these: 48, 59; 1 x 14336 x 4096: 22.5, 26; 8 of these: 24.6, 26.6; 16: 29, 26.
// With norm and unit, 1 x 4096 x 28672: 46, beside 72 for three kernels.

#include "hip_common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));


struct LinearFewArgs {
  const __bf16 *x, *w, *bias, *res, *norm;
  __bf16* y;
  int M, O, K;             // O: columns of y
  long ldx, ldw, ldr, ldy;
  float eps, offset;       // norm weights are norm + offset
};

enum { LF_PLAIN = 0, LF_SILU = 1, LF_GELU = 2 };

// RT tiles of 16 rows of W; with a gated unit half of them are the gate's, the
// others the up projection's
template <int RT, int ACT, bool NORM, int NW, int U>
__global__ __launch_bounds__(NW * WAVE) void linear_few_kernel(
    const LinearFewArgs a) {
    __shared__ __attribute__((aligned(16))) f32x4 red[NW][RT][WAVE];
  __shared__ float squares[NORM ? NW : 1][WAVE];

  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int l16 = lane & 15, lg = lane >> 4;
  constexpr int YT = ACT ? RT / 2 : RT;  // tiles of y's columns
  const int row0 = blockIdx.x * 16 * YT;

  const __bf16* wp[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int row = r / YT * a.O + min(row0 + r % YT * 16 + l16, a.O - 1);
    wp[r] = a.w + (long)row * a.ldw + lg * 8;
  }
  const __bf16* xp = a.x + (long)min(l16, a.M - 1) * a.ldx + lg * 8;

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

  const int steps = a.K / 32, chunks = steps / U;
  // operands of one chunk; the next one's are asked for before this one is used,
  // rows of x among them, as loads come back in order
  struct Chunk {
    bf16x8_t w[RT][U], x[U], g[NORM ? U : 1];
  };
  auto fetch = [&](Chunk& f, int c) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int at = (c * U + u) * 32;
#pragma unroll
      for (int r = 0; r < RT; ++r) f.w[r][u] = load(wp[r] + at);
      f.x[u] = load(xp + at);
      if (NORM) f.g[u] = load(a.norm + at + lg * 8);
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
  Chunk one, two;
  if (wid < chunks) fetch(one, wid);
  for (int c = wid; c < chunks; c += 2 * NW) {
    if (c + NW < chunks) fetch(two, c + NW);
    use(one);
    if (c + 2 * NW < chunks) fetch(one, c + 2 * NW);
    if (c + NW < chunks) use(two);
  }
  // steps that make no whole chunk
  for (int s = chunks * U + wid; s < steps; s += NW) {
    bf16x8_t v = load(xp + s * 32);
    if (NORM) v = normed(v, load(a.norm + s * 32 + lg * 8));
#pragma unroll
    for (int r = 0; r < RT; ++r)
      acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load(wp[r] + s * 32), v,
                                                       acc[r], 0, 0, 0);
  }

#pragma unroll
  for (int r = 0; r < RT; ++r) red[wid][r][lane] = acc[r];
  if (NORM) squares[wid][lane] = sq;
  __syncthreads();

  // a wave per tile of y: four columns of a row a lane
  for (int r = wid; r < YT; r += NW) {
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
    const int row = l16, col = row0 + r * 16 + lg * 4;
    if (row >= a.M) continue;
    float o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int at = min(col + j, a.O - 1);
      float f = v[0][j];
      if (ACT) {
        float up = v[1][j];
        if (a.bias) {
          f += (float)a.bias[at];
          up += (float)a.bias[a.O + at];
        }
        if (ACT == LF_SILU) {
          f = f / (1.0f + __expf(-f)) * up;
        } else {
          const float z = 0.7978845608028654f * (f + 0.044715f * f * f * f);
          f = 0.5f * f * (1.0f + tanhf(z)) * up;
        }
      } else if (a.bias) {
        f += (float)a.bias[at];
      }
      if (a.res) f += (float)a.res[(long)row * a.ldr + at];
      o[j] = f;
    }
    __bf16* y = a.y + (long)row * a.ldy + col;
    if (col + 3 < a.O && a.ldy % 4 == 0) {
      typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
      *reinterpret_cast<bf16x4_t*>(y) =
          bf16x4_t{(__bf16)o[0], (__bf16)o[1], (__bf16)o[2], (__bf16)o[3]};
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (col + j < a.O) y[j] = (__bf16)o[j];
    }
  }
}

template <int RT, int ACT, int NW, int U>
static void linear_few_go(const LinearFewArgs& a, hipStream_t stream) {
  constexpr int cols = 16 * (ACT ? RT / 2 : RT);
  const dim3 grid((unsigned)((a.O + cols - 1) / cols)), block(NW * WAVE);
  // the norm's weights and sums need registers: shorter chunks
  if (a.norm) {
    linear_few_kernel<RT, ACT, true, NW, 2><<<grid, block, 0, stream>>>(a);
  } else {
    linear_few_kernel<RT, ACT, false, NW, U><<<grid, block, 0, stream>>>(a);
  }
}

// Tiles of W's rows per block: one up to 4096 rows, which are 256 blocks; two up
// to 8192 (6144 rows, 16 of x: 13.7 us, 17.0 with one); beyond that four, where
// rows of x are read once for 64 of W (28672 rows, 16 of x: 48 us, 51 with two, 56
// with one), but one for few rows of x (one: 38 us, 45 with four).  A unit needs
// both its halves; four from 16384 rows on (28672 rows, 16 of x, norm: 50 us, 53
// with two; 12800, one of x: 14.0 with two, 15.8).
static void linear_few_tiles(const LinearFewArgs& a, int act, hipStream_t stream) {
  if (act == LF_SILU) {
    if (a.O >= 8192) linear_few_go<4, LF_SILU, 4, 2>(a, stream);
    else linear_few_go<2, LF_SILU, 8, 4>(a, stream);
  } else if (act == LF_GELU) {
    if (a.O >= 8192) linear_few_go<4, LF_GELU, 4, 2>(a, stream);
    else linear_few_go<2, LF_GELU, 8, 4>(a, stream);
  } else if (a.O <= 4096 || (a.O > 8192 && a.M <= 4)) {
    linear_few_go<1, LF_PLAIN, 8, 4>(a, stream);
  } else if (a.O <= 8192) {
    linear_few_go<2, LF_PLAIN, 8, 4>(a, stream);
  } else {
    linear_few_go<4, LF_PLAIN, 4, 2>(a, stream);
  }
}

// Strides in elements; 16-byte loads: x, w, norm and the strides of x and w are
// multiples of 8 elements, K of 32.  M up to 16.
extern "C" void launch_linear_few(const void* x, const void* w, const void* bias,
                                  const void* res, const void* norm, void* y,
                                  int M, int O, int K, long ldx, long ldw,
                                  long ldr, long ldy, float eps, float offset,
                                  int act, hipStream_t stream) {
  const LinearFewArgs a{(const __bf16*)x, (const __bf16*)w, (const __bf16*)bias,
                        (const __bf16*)res, (const __bf16*)norm, (__bf16*)y,
                        M, O, K, ldx, ldw, ldr, ldy, eps, offset};
  linear_few_tiles(a, act, stream);
}
