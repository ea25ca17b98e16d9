// A block of a product whose waves have rings of their own (linear_own.hip), for the kernels
// that are made of it.
#pragma once

#include <type_traits>

#include "linear_few_kernel.h"

namespace {

constexpr int OWN_WAVES = 8;
constexpr int OWN_LDS = 150 * 1024;  // that rings may take, beside squares

template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// Waits until at most the loads of the `younger` last chunks, PER each, are under way; J: of
// how many that may be at most.
template <int J, int PER>
__device__ __forceinline__ void wait_chunks(int younger) {
  if constexpr (J == 0) {
    wait_loads<0>();
  } else {
    if (younger >= J) wait_loads<J * PER>();
    else wait_chunks<J - 1, PER>(younger);
  }
}

// A barrier for loads to LDS on either side of it: this wave's reads of LDS have returned, so that
// other waves may load into their places.
__device__ __forceinline__ void meet() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

__device__ __forceinline__ unsigned lds_at(const char* smem) {
  return (unsigned)(unsigned long long)(const __attribute__((address_space(3))) char*)smem;
}

// How a tile's sixteen rows lie in W.  GATED: a tile has eight columns, rows 4g and 4g + 1 are
// the gate's of columns 2g and 2g + 1, the two others the up projection's, O rows behind them, so
// that a lane has both sums of a column.  TURNED: the same with the two dimensions that a rotation
// takes, n_zero apart (half a head, a power of two); O counts them as one.
// CLAMPED: GATED with the clamped unit, which as a branch of the others costs them 1 to 2 us in a
// step of 530.
enum { APART = 0, GATED_ROWS = 1, TURNED_ROWS = 2, CLAMPED_ROWS = 3 };
template <int ROWS>
__device__ __forceinline__ const __bf16* row_of(const LinearFewArgs& a, int col0, int row) {
  if (ROWS == APART) return a.w + (long)min(col0 + row, a.O - 1) * a.ldw;
  const int t = row >> 4, q = row & 15;
  const int col = min(col0 + t * 8 + (q >> 2) * 2 + (q & 1), a.O - 1);
  if (ROWS == TURNED_ROWS)
    return a.w + (long)(2 * col - (col & (a.n_zero - 1)) + (q & 2 ? a.n_zero : 0)) * a.ldw;
  return a.w + (long)((q & 2 ? a.O : 0) + col) * a.ldw;
}

// A block's place among those of W's rows, and its first row of x, of which it has `rows`:
// blocks of the same rows of W are eight apart.
struct BlockPlace {
  int bx, x0;
};
__device__ __forceinline__ BlockPlace place_of(const LinearFewArgs& a, int rows, int block) {
  const int groups = (a.M + rows - 1) / rows;
  if (groups == 1) return {block, 0};
  const int pack = block >> 3;
  return {pack / groups * 8 + (block & 7), pack % groups * rows};
}

// a tile's sums to memory (gated: act(gate) * up of two columns); parts: the unit
template <int GATED>
__device__ __forceinline__ void finish_tile(const LinearFewArgs& a, int row, int col0, int lg,
                                            const f32x4& v, const Ends<0>& e) {
  if (!GATED) {
    finish_columns<LF_PLAIN>(a, row, col0 + lg * 4, &v, e);
    return;
  }
  const int col = col0 + lg * 2;
  float o[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int at = min(col + j, a.O - 1);
    float f = v[j], up = v[j + 2];
    if (GATED == CLAMPED_ROWS) {
      if (a.bias && at < a.n_zero) f += (float)a.bias[at], up += (float)a.res[at];
    } else if (a.bias) {
      f += (float)a.bias[at], up += (float)a.bias[a.O + at];
    }
    if (GATED == CLAMPED_ROWS) {
      f = fminf(f, a.eps);
      f = f / (1.0f + __expf(-a.offset * f)) * (fminf(fmaxf(up, -a.eps), a.eps) + 1.0f);
    } else if (a.parts == LF_SILU) {
      f = f / (1.0f + __expf(-f)) * up;
    } else {
      const float z = 0.7978845608028654f * (f + 0.044715f * f * f * f);
      f = 0.5f * f * (1.0f + tanhf(z)) * up;
    }
    if (GATED != CLAMPED_ROWS && a.res) f += (float)a.res[(long)row * a.ldr + at];
    o[j] = f;
  }
  __bf16* y = a.y + (long)row * a.ldy + col;
  if (col + 1 < a.O && a.ldy % 2 == 0) {
    *reinterpret_cast<bf16x2_t*>(y) = bf16x2_t{(__bf16)o[0], (__bf16)o[1]};
  } else {
#pragma unroll
    for (int j = 0; j < 2; ++j)
      if (col + j < a.O) y[j] = (__bf16)o[j];
  }
}

// What a wave's rows of x become with the norm's weights, and their squares.
__device__ __forceinline__ bf16x8_t times(bf16x8_t v, bf16x8_t g, float offset, float& sq) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float f = (float)v[j];
    sq = fmaf(f, f, sq);
    v[j] = (__bf16)(f * ((float)g[j] + offset));
  }
  return v;
}

// The sums of all shares of a tile of `steps` of the contraction, times the norm's factor.
template <int TT, int SHARES, int TW, bool NORM>
__device__ __forceinline__ f32x4 sum_of(const LinearFewArgs& a, const f32x4* red,
                                        const float (*squares)[TW][WAVE], int tiles, int n,
                                        int lane) {
  const int i = n % TT;
  f32x4 v{0, 0, 0, 0};
#pragma unroll
  for (int p = 0; p < SHARES; ++p) {
    const f32x4 f = red[(p * tiles + n) * WAVE + lane];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] += f[j];
  }
  if (NORM) {
    float s = 0.0f;
#pragma unroll
    for (int p = 0; p < SHARES; ++p) s += squares[i / TW * SHARES + p][i % TW][lane];
    s += __shfl_xor(s, 16, WAVE);
    s += __shfl_xor(s, 32, WAVE);
    const float f = rsqrtf(s / a.K + a.eps);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] *= f;
  }
  return v;
}

// Rows of 32 bits that are added to four columns of a row of y (PAIRS), asked for as Ends are:
// the first eight stay in registers.
struct PairRows {
  f32x4 first[8];
  const float* rest;
  long ld;

  __device__ __forceinline__ void read(const LinearFewArgs& a, int row, int col) {
    ld = a.O;
    rest = a.part + (long)min(row, a.M - 1) * a.n_zero * ld + min(col, a.O - 4);
#pragma unroll
    for (int k = 0; k < 8; ++k)
      first[k] = *reinterpret_cast<const f32x4*>(rest + min(k, a.n_zero - 1) * ld);
  }
  __device__ __forceinline__ void add(f32x4& v, int n) const {
    f32x4 sum = first[0];
#pragma unroll
    for (int k = 1; k < 8; ++k)
      if (k < n) sum += first[k];
    for (int k = 8; k < n; ++k) sum += *reinterpret_cast<const f32x4*>(rest + k * ld);
    v += sum;
  }
};

// RT, TT: tiles of 16 rows of W and of x; SL: chunks of a wave under way.  The norm's weights
// lie in LDS, all of them.  SHARED: blocks have a share of a contraction each.  PAIRS: to a
// row of y, n_zero rows of `part` are added, which lie side by side (no norm, no share).
// finish: what becomes of a tile's sums (finish_tile).
template <int RT, int TT, int SL, int GATED, bool NORM, bool SHARED, bool PAIRS, typename F>
__device__ __forceinline__ void own_block(const LinearFewArgs& a, int block, F finish) {
  constexpr int LOADS = (RT + TT) * 2, CHUNK = LOADS * 1024;
  constexpr int COLS = (GATED ? 8 : 16) * RT;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ float squares[NORM ? OWN_WAVES : 1][TT][WAVE];

  arrive(a);
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int l16 = lane & 15, lg = lane >> 4;
  const BlockPlace place = place_of(a, 16 * TT, block);
  const int bx = place.bx, x0 = place.x0, col0 = bx * COLS;
  if (col0 >= a.O) return;

  // A load is 8 rows of 128 bytes.  Pieces of a row are swapped by the row, so that those
  // that a read meets lie in different banks.
  const char* from[LOADS];
  int col[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) col[i] = ((lane & 7) ^ ((i * 8 + (lane >> 3)) & 7)) * 8;
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = i * 8 + (lane >> 3);
    from[i] = (const char*)(i < RT * 2
                                ? row_of<GATED>(a, col0, row)
                                : a.x + (long)min(x0 + row - RT * 16, a.M - 1) * a.ldx);
  }
  const int c0 = SHARED ? blockIdx.y * a.share : 0;
  const int all = (a.K + 63) / 64 - c0, chunks = SHARED ? min(a.share, all) : all;
  const int first = first_of(a, a.share, chunks, bx);
  const int mine = wid < chunks ? (chunks - 1 - wid) / OWN_WAVES + 1 : 0;
  auto chunk = [&](int n) {
    const int c = wid + n * OWN_WAVES + first;
    return c0 + (c >= chunks ? c - chunks : c);
  };
  const int ring = wid * SL * CHUNK;
  const unsigned lds = lds_at(smem);
  auto issue = [&](int n, int slot) {
    const int k0 = chunk(n) * 64;
    unsigned k[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) k[i] = (unsigned)min(k0 + col[i], a.K - 8) * 2;
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      to_lds(from[i] + k[i & 1], lds + ring + slot * CHUNK + i * 1024);
  };
  constexpr int G = OWN_WAVES * SL * CHUNK;  // where the norm's weights lie
  if (NORM) {
    for (int i = wid; i * 512 < a.K; i += OWN_WAVES)
      to_lds((const char*)(a.norm + min(i * 512 + lane * 8, a.K - 8)), lds + G + i * 1024);
  }
#pragma unroll
  for (int s = 0; s < SL; ++s)
    if (s < mine) issue(s, s);

  f32x4 acc[RT][TT];
  float sq[TT];
#pragma unroll
  for (int i = 0; i < TT; ++i) {
    sq[i] = 0.0f;
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[r][i] = f32x4{0, 0, 0, 0};
  }
  if (NORM) {
    wait_chunks<SL, LOADS>(mine);
    meet();
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
  PairRows pairs[PAIRS ? TILES : 1];
  if (PAIRS) {
#pragma unroll
    for (int q = 0; q < TILES; ++q) {
      const int n = min(wid + q * OWN_WAVES, RT * TT - 1);
      pairs[q].read(a, x0 + n % TT * 16 + l16, col0 + n / TT * 16 + lg * 4);
    }
  }
  int slot = 0;
  for (int n = 0; n < mine; ++n) {
    wait_chunks<SL - 1, LOADS>(mine - 1 - n);
    const int k0 = chunk(n) * 64;
    const char* at = smem + ring + slot * CHUNK + l16 * 128;
    bf16x8_t w[RT][2], v[TT][2], g[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int piece = ((u * 4 + lg) ^ (l16 & 7)) * 16;
#pragma unroll
      for (int i = 0; i < TT; ++i)
        v[i][u] = *reinterpret_cast<const bf16x8_t*>(at + (RT + i) * 2048 + piece);
      if (NORM)
        g[u] = *reinterpret_cast<const bf16x8_t*>(smem + G + (k0 + u * 32 + lg * 8) * 2);
#pragma unroll
      for (int r = 0; r < RT; ++r)
        w[r][u] = *reinterpret_cast<const bf16x8_t*>(at + r * 2048 + piece);
    }
    // all read: the chunk's place is free
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (n + SL < mine) issue(n + SL, slot);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (u && k0 + 32 >= a.K) break;  // K is a multiple of 32
#pragma unroll
      for (int i = 0; i < TT; ++i) {
        const bf16x8_t x = NORM ? times(v[i][u], g[u], a.offset, sq[i]) : v[i][u];
#pragma unroll
        for (int r = 0; r < RT; ++r)
          acc[r][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[r][u], x, acc[r][i], 0, 0, 0);
      }
    }
    if (++slot == SL) slot = 0;
  }
  __syncthreads();
  f32x4* red = reinterpret_cast<f32x4*>(smem);  // [waves][RT][TT][lanes]
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int i = 0; i < TT; ++i) red[((wid * RT + r) * TT + i) * WAVE + lane] = acc[r][i];
  if (NORM) {
#pragma unroll
    for (int i = 0; i < TT; ++i) squares[wid][i][lane] = sq[i];
  }
  __syncthreads();

  if (a.zero && block == 0)
    for (int i = threadIdx.x; i < a.n_zero; i += OWN_WAVES * WAVE) a.zero[i] = 0;
#pragma unroll
  for (int q = 0; q < TILES; ++q) {
    const int n = wid + q * OWN_WAVES;
    if (n >= RT * TT) break;
    f32x4 v = sum_of<TT, OWN_WAVES, TT, NORM>(a, red, squares, RT * TT, n, lane);
    if (SHARED && !sums_of_all(a, (long)bx * RT * TT + n, lane, v)) continue;
    const int row = x0 + n % TT * 16 + l16;
    if (PAIRS) pairs[q].add(v, a.n_zero);
    if (row < a.M)
      finish(row, col0 + n / TT * (GATED ? 8 : 16), lg, v, ends[q]);
  }
}
template <int RT, int TT, int SL, int GATED, bool NORM, bool SHARED, bool PAIRS>
__device__ __forceinline__ void own_block(const LinearFewArgs& a, int block) {
  own_block<RT, TT, SL, GATED, NORM, SHARED, PAIRS>(
      a, block, [&](int row, int col, int lg, const f32x4& v, const Ends<0>& e) {
        finish_tile<GATED>(a, row, col, lg, v, e);
      });
}

// columns: of a chunk or stage
inline void turned(LinearFewArgs& a, int act, int columns) {
  a.parts = (unsigned char)act;
  a.share = (a.K + columns - 1) / columns;
  a.turn = a.share > 1 && in_step(a.ldw)
               ? (unsigned)(((1ull << 32) + a.share - 1) / a.share) : 0;
}

// LDS of a block; slots: chunks of a wave
constexpr int own_room(int rt, int tt, int slots, int K, bool norm) {
  const int ring = OWN_WAVES * slots * (rt + tt) * 2048 + (norm ? (K + 511) / 512 * 1024 : 0);
  const int sums = OWN_WAVES * rt * tt * 1024;
  return ring > sums ? ring : sums;
}

// Tiles of W's rows and of x's for M rows and `tiles`, beside `others` blocks, in kernels
// that take no more than four of W's: as for other products (linear_own.hip).
struct Tiles {
  int rt, tt, blocks;
};
inline Tiles tiles_beside(int M, int tiles, int others, int K, bool norm) {
  Tiles best{0, 0, 0};
  long least = 0;
  const int whole = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  for (int rt = 1; rt <= 4; ++rt)
    for (int tt = whole; tt && tt * 2 >= whole; tt /= 2) {
      // (one tile of W and 64 rows of x: as in linear_own.hip)
      if ((rt == 1 && tt == 4) || own_room(rt, tt, 1, K, norm) > OWN_LDS) continue;
      const int groups = (M + 16 * tt - 1) / (16 * tt);
      int blocks = (tiles + rt - 1) / rt;
      if (groups > 1) blocks = (blocks + 7) / 8 * 8 * groups;
      const long reads = (long)((blocks + others + 255) / 256) *
                         (M > 16 ? 2 * (rt + tt) : 2 * rt + 1);
      if (!best.rt || reads < least || (reads == least && tt < best.tt))
        best = {rt, tt, blocks}, least = reads;
    }
  return best;
}

// f with the constants rt and tt
template <typename F>
void with_tiles(const Tiles& t, F f) {
  switch (t.rt * 8 + t.tt) {
#define CASE(R, T) \
  case R * 8 + T: f(std::integral_constant<int, R>(), std::integral_constant<int, T>()); break;
    CASE(1, 1) CASE(2, 1) CASE(3, 1) CASE(4, 1)
    CASE(1, 2) CASE(2, 2) CASE(3, 2) CASE(4, 2)
    CASE(2, 4) CASE(3, 4) CASE(4, 4)
#undef CASE
  }
}

}  // namespace
