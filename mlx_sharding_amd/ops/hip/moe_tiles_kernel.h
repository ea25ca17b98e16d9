// Products of routed experts over tiles of one expert's (token, expert) pairs.
//
// What bounds them: the matrix cores, and the power that they draw (clocks of 1.7 to 1.8
// GHz).  A block of four waves makes 256 pairs by 256 rows of weights, a wave 128 x 128,
// whose sums fill the accumulation registers: a stage of 64 columns then takes 2048 cycles
// of every core and half as many of LDS.  Rows of 64 columns are whole lines of 128 bytes
// (of 32 columns twice as many requests), and pieces of 16 bytes within a row are swapped
// by the row, so that rows that a read meets lie in different banks.  LDS holds two
// stages; a wave works on one by quarters, and each half of its operands is replaced by
// loads of the stage after the next as soon as all waves have read it.  More than three
// instructions between two products hold up the second, and so do loads that come in one
// run: loads and LDS reads stand alone between products, eight apart, with addresses that
// need one scalar sum.  A block walks over its tiles without a gap: behind a tile's last
// stage come the next one's, and results are stored meanwhile.
// Products of 16 x 16 x 32 move half as many sums per operation as those of 32 x 32 x 16:
// at one share of busy cores clocks are 7% higher.
// Measured: 32768 tokens, top 6 of 64 experts, 2048 -> 1408: 2.02 -> 1.80 ms (1260
// TFLOP/s), 1408 -> 2048: 1.20 -> 1.03 (1100), before with a ring of four stages of 32
// columns; one wait for a stage's loads, all in its middle: 1.92 and 1.11.  Without loads
// the cores are 78% busy, without loads and reads 83, as it is 74.  Contractions of two to
// five stages pay for the first one's size: both products up to 1.3 us more than with 32
// columns (8 experts of 128 x 128 25.1 -> 26.2 us, 90 of 320 x 192 35.8 -> 37.1).
// Clamped units read their pairs' weights out of LDS at the end of an item, where a load
// from memory would wait for the stages under way.
#pragma once

#include "moe_tiles.h"

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// s_waitcnt for at most n loads and stores and r LDS reads under way
constexpr int vm_wait(int n, int r) { return (n & 15) | 0x70 | r << 8 | (n >> 4) << 14; }

#define MT_GROUP 4  // tiles whose blocks run together, with the same weights
// MT: pairs of a tile.  DENSE: of one matrix, whose pairs are the rows of x; blocks may
// have shares of the contraction each.  R: stages that LDS holds; an item has as many.
template <int MT, MoeUnit UNIT, int R, bool DENSE>
__global__ __launch_bounds__(256, 1) void moe_tiles_kernel(const MoeTilesArgs a) {
#ifdef __HIP_DEVICE_COMPILE__  // buffer resources are no type of the host's
  constexpr bool PARTS = UNIT == MT_PARTS;
  constexpr bool GLU = UNIT != MT_SUMS && UNIT != MT_PARTS;
  constexpr bool GATHERED = GLU && !DENSE;  // rows of x by the pairs' tokens
  constexpr int NX = MT / 32;           // 16-pair tiles of a wave, rows of x it brings in 8
  constexpr int L = 8 + NX, LH = L / 2;  // loads per wave and stage, and half a stage
  constexpr int ST = (256 + MT) * 128;  // bytes of a stage
  constexpr int NC = GLU ? 128 : 256;   // outputs of a block
  // a wave's, of an item (of sums in 32 bits: too many to wait for less than all)
  constexpr int STORES = PARTS ? 0 : NX * NC / 64;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wid >> 1, wn = wid & 1;
  const int stages = a.K / 64;

  // an XCD has consecutive tiles, its blocks walk them in groups
  const int total = DENSE ? (a.rows + MT - 1) / MT : *a.n_tiles;
  const int group = DENSE ? min(total, MT_GROUP)
                    : total >= 16 * MT_GROUP ? MT_GROUP : 1;  // few: to all XCDs
  const int items = total * a.cols * a.shares;  // dense
  const int per = DENSE ? (items + 7) / 8 : (total + 8 * group - 1) / (8 * group) * group;
  const int xcd = blockIdx.x & 7, step = gridDim.x >> 3;
  int slot = (int)(blockIdx.x >> 3) - step;
  struct Item { int e, p0, np, n0, share, k0, n; };  // n: stages, from k0 on
  struct Place { int tile, n0, share; };  // a tile, or -1 behind the last one
  auto advance = [&]() -> Place {
    for (;;) {
      slot += step;
      if constexpr (DENSE) {
        const int at = xcd * per + slot;
        if (slot >= per || at >= items) return {-1, 0, 0};
        const int share = at / (total * a.cols), in = at % (total * a.cols);
        const int grp = in / (group * a.cols), rest = in % (group * a.cols);
        const int tiles = min(group, total - grp * group);
        return {grp * group + rest % tiles, rest / tiles * NC, share};
      }
      const int grp = slot / (group * a.cols), rest = slot % (group * a.cols);
      const int ti = grp * group + rest % group;
      if (ti >= per) return {-1, 0, 0};
      if (xcd * per + ti < total) return {xcd * per + ti, rest / group * NC, 0};
    }
  };
  // a tile's entry is read by scalar loads: what vector loads bring to registers would
  // be waited for with all stages under way (tokens and weights go to LDS)
  auto item = [&](const Place& at) -> Item {
    const int tile = max(at.tile, 0);
    if constexpr (DENSE) {
      const int k0 = at.share * stages / a.shares, k1 = (at.share + 1) * stages / a.shares;
      return {0, tile * MT, min(MT, a.rows - tile * MT), at.n0, at.share, k0, k1 - k0};
    }
    const auto* t = (const __attribute__((address_space(4))) int*)a.tiles + tile * 3;
    return {t[0], t[1], t[2], at.n0, 0, 0, stages};
  };
  // A wave's rows of a stage: of the weights, of which a load brings rows WR behind those
  // of the load before (behind the last rows the last ones again: O is a multiple of 64),
  // the first and the last load's; of x, each lane's.  Of a gated unit, waves 0 and 1
  // bring gate rows, 2 and 3 up rows (16 by turns).
  constexpr unsigned WR = GLU ? 16 : 32;
  struct Rows { const char *w, *x; unsigned w_off, w_at[8], off[NX]; };
  auto pair_of = [&](const Item& it, int i) {
    return min((i * 4 + wid) * 8 + (lane >> 3), it.np - 1);
  };
  // t: rows of x
  auto rows_of = [&](const Item& it, const int (&t)[NX], Rows& s) {
    const unsigned at = ((lane & 7) ^ (lane >> 3)) * 16;
    s.w = (GLU && wid >> 1 ? a.w2 : a.w) + it.e * a.wstride + (long)it.n0 * a.ldw +
          it.k0 * 128;
    s.x = a.x + (GATHERED ? 0 : it.p0 * a.xstride) + it.k0 * 128;
    s.w_off = ((GLU ? wid & 1 : wid) * 8 + (lane >> 3)) * a.ldw + at;
#pragma unroll
    for (int i = 0; i < 8; ++i) s.w_at[i] = min(i * WR, a.O - WR - it.n0) * a.ldw;
#pragma unroll
    for (int i = 0; i < NX; ++i) s.off[i] = (unsigned)t[i] * (unsigned)a.xstride + at;
  };
  // the i-th of the loads of a stage, to its place in LDS
  auto load = [&](const Rows& s, __amdgpu_buffer_rsrc_t w, __amdgpu_buffer_rsrc_t x, int at,
                  int i) {
    auto* to = (__attribute__((address_space(3))) void*)(smem + at + (i * 4 + wid) * 1024);
    if (i < 8) __builtin_amdgcn_raw_ptr_buffer_load_lds(w, to, 16, s.w_off, s.w_at[i], 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(x, to, 16, s.off[i - 8], 0, 0, 0);
  };
  // the k-th stage
  auto columns = [](const char* p, int k) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)(p + k * 128), 0, -1, 0x00027000);
  };
  // numbers that belong to an item's pairs, into LDS
  auto numbers = [&](const void* of, const Item& it, char* to) {
    if (wid * 64 < MT)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(
              (const int*)of + it.p0 + min(wid * 64 + lane, it.np - 1)),
          (__attribute__((address_space(3))) void*)(to + wid * 256), 4, 0, 0);
  };
  // read here: the compiler would wait for all loads to LDS
  auto number = [](const char* at) {
    int v;
    asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(v)
                 : "v"((const __attribute__((address_space(3))) char*)at) : "memory");
    return v;
  };
  char* const next_tokens = smem + R * ST;
  Place at = advance();
  if (at.tile < 0) return;
  Item it = item(at);
  at = advance();
  Rows rows;
  {
    int tok[NX];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      tok[i] = pair_of(it, i);
      if (GATHERED) tok[i] = a.tokens[it.p0 + tok[i]];
    }
    rows_of(it, tok, rows);
  }

  // A stage is worked on by quarters: halves of a wave's rows of weights by halves of its
  // rows of x.  Operands of a half are w[half][tile][columns / 32], x likewise.
  constexpr int HX = NX / 2;
  f32x4 acc[8][NX];
  bf16x8_t w[2][4][2], x[2][HX][2];
  const int l16 = lane & 15;
  const int wo = (wn * 128 + l16) * 128, xo = (256 + wm * (MT / 2) + l16) * 128;
  const int at16[2] = {((lane >> 4) ^ (l16 & 7)) * 16, ((lane >> 4 | 4) ^ (l16 & 7)) * 16};
  auto rd = [](const char* p) { return *reinterpret_cast<const bf16x8_t*>(p); };
  // the r-th operand of a half
  auto read_w = [&](int at, int h, int r) {
    w[h][r >> 1][r & 1] =
        rd(smem + at + at16[r & 1] + wo + (h * 4 + (r >> 1)) * 2048);
  };
  auto read_x = [&](int at, int h, int r) {
    x[h][r >> 1][r & 1] =
        rd(smem + at + at16[r & 1] + xo + (h * HX + (r >> 1)) * 2048);
  };
  // the c-th load of a half: a wave's share of w[h] and x[h] of all waves
  auto load_half = [&](const Rows& s, __amdgpu_buffer_rsrc_t sw, __amdgpu_buffer_rsrc_t sx,
                       int at, int h, int c) {
    constexpr int Q = NX / 4;
    if (c < 4) load(s, sw, sx, at, (c >> 1) * 4 + h * 2 + (c & 1));
    else load(s, sw, sx, at, 8 + (c - 4) / Q * 2 * Q + h * Q + (c - 4) % Q);
  };
#pragma unroll
  for (int k = 0; k < R; ++k)
#pragma unroll
    for (int c = 0; c < L; ++c)
      load_half(rows, columns(rows.w, k), columns(rows.x, k), k * ST, c / LH, c % LH);
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"((R - 1) * L) : "memory");
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int r = 0; r < 8; ++r) read_w(0, 0, r);
#pragma unroll
  for (int r = 0; r < NX; ++r) read_x(0, 0, r);

  int here = 0, after = ST;  // places of this stage and the next one
  int flip = 0;
  int lax = 0;  // meetings behind all of an item's stores
  for (bool more = true; more;) {
    more = at.tile >= 0;
    const Item nx = more ? item(at) : it;
    if (more) at = advance();
    // read R stages before this item's end, when a meeting has waited for them
    if constexpr (GATHERED) numbers(a.tokens, nx, next_tokens);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < NX; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0f;
    // weights of this item's pairs go to LDS, and are there some steps later; those of
    // the item before may still be read
    if constexpr (UNIT == MT_CLAMPED) {
      flip ^= 1;
      numbers(a.scale, it, next_tokens + (1 + flip) * MT * 4);
    }
    // A stage's products; between them, one at a time and evenly, operands of the quarter
    // behind, and loads of the R-th stage from here.  Loads replace a half when all waves
    // have read it (they meet twice a stage, in the middle of a quarter, where nobody
    // waits for an operand), and are read three quarters of a stage later at least.
    auto between = [&](int m, __amdgpu_buffer_rsrc_t sw, __amdgpu_buffer_rsrc_t sx) {
      constexpr int Q = 4 * NX, EACH = NX / 4;  // products of a quarter, from read to read
      const int r = m % Q / EACH;
      const bool now = m % EACH == 0;
      if (m < Q && now && r < NX) read_x(here, 1, r);
      if (m / Q == 1 && now && r < 8) read_w(here, 1, r);
      if (m / Q == 2 && now && r < 8) read_w(after, 0, r);
      if (m / Q == 3) {  // behind the last product of the one that it replaces
        const int n = m - 3 * Q;
        if (n % 8 == 7 || (n % 8 == 0 && n)) read_x(after, 0, n / 4 - 1);
        if (n == Q - 1) read_x(after, 0, NX - 1);
      }
#pragma unroll
      for (int c = 0; c < LH; ++c) {
        if (m == Q / 2 + 1 + c * (2 * Q / LH)) load_half(rows, sw, sx, here, 0, c);
        if (m == 5 * Q / 2 + 1 + c * (3 * Q / 2 / LH)) load_half(rows, sw, sx, here, 1, c);
      }
      if (m == Q / 2 - 1 || m == 5 * Q / 2 - 1) {
        // an item's stores came behind these loads and need not be done
        constexpr int READS = NX < 8 ? NX : 8, AWAY = (2 * R - 3) * LH;
        __builtin_amdgcn_s_waitcnt(vm_wait(AWAY + STORES, READS));
        if (__builtin_expect(lax <= 0, 1)) __builtin_amdgcn_s_waitcnt(vm_wait(AWAY, READS));
        asm volatile("s_barrier" ::: "memory");
        --lax;
      }
    };
    auto stage = [&](int k) {
      const auto sw = columns(rows.w, k), sx = columns(rows.x, k);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int hw = q >> 1, hx = (q ^ q >> 1) & 1;
#pragma unroll
        for (int j = 0; j < HX; ++j)
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              f32x4& to = acc[hw * 4 + t][hx * HX + j];
              to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[hw][t][c], x[hx][j][c], to, 0, 0, 0);
              __builtin_amdgcn_sched_barrier(0);
              between(((q * HX + j) * 2 + c) * 4 + t, sw, sx);
              __builtin_amdgcn_sched_barrier(0);
            }
      }
      here = after;
      after = R == 2 ? after ^ ST : after == (R - 1) * ST ? 0 : after + ST;
    };
    if (GATHERED && stages < 2 * R) asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    int k = R;
    for (int left = it.n - R, part = 0; part < 2; left = R, ++part) {
      if (part) {  // behind the last stage of this item come the next one's
        k = 0;
        int tok[NX];
#pragma unroll
        for (int i = 0; i < NX; ++i) {
          tok[i] = pair_of(nx, i);
          if (GATHERED) tok[i] = number(next_tokens + tok[i] * 4);
        }
        rows_of(nx, tok, rows);
      }
      for (; left > 0; --left, ++k) stage(k);
    }
    __builtin_amdgcn_sched_barrier(0);
    // sums are taken out of the accumulation registers one by one: read by the
    // compiler, all are copied at once, more than there are registers for.  It does
    // not know what reads them here, so the wait for the last products is written out.
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    auto sum = [&](int i, int j, int r) {
      float v;
      asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(acc[i][j][r]));
      return v;
    };
    // lane: pair l16, outputs 4 (lane / 16) .. + 3 of 16; of two such runs, lanes get 8
    // outputs side by side
    auto store = [&](__bf16* row, int o, const float (&lo)[4], const float (&up)[4]) {
      u32x2 x, y;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        x[h] = __builtin_bit_cast(unsigned, bf16x2_t{(__bf16)lo[2 * h], (__bf16)lo[2 * h + 1]});
        y[h] = __builtin_bit_cast(unsigned, bf16x2_t{(__bf16)up[2 * h], (__bf16)up[2 * h + 1]});
      }
      const auto s0 = __builtin_amdgcn_permlane16_swap(x[0], y[0], false, false);
      const auto s1 = __builtin_amdgcn_permlane16_swap(x[1], y[1], false, false);
      o += (lane >> 4 & 1) * 16 + (lane >> 5) * 8;
      if (o < a.O) *reinterpret_cast<u32x4*>(row + o) = u32x4{s0[0], s1[0], s0[1], s1[1]};
    };
    if constexpr (PARTS) {
      // rows behind the last pair repeat it
#pragma unroll
      for (int j = 0; j < NX; ++j) {
        const int p = min(wm * (MT / 2) + j * 16 + l16, it.np - 1);
        float* row = a.parts + ((long)it.share * a.rows + it.p0 + p) * a.O;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int o = it.n0 + wn * 128 + i * 16 + (lane >> 4) * 4;
          const f32x4 v = {sum(i, j, 0), sum(i, j, 1), sum(i, j, 2), sum(i, j, 3)};
          if (o < a.O) *reinterpret_cast<f32x4*>(row + o) = v;
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    } else {
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      const int p = wm * (MT / 2) + j * 16 + l16;
      // all lanes take part in the exchange
      __bf16* row = a.y + (long)(it.p0 + min(p, it.np - 1)) * a.O;
      float by = 1.0f;
      if constexpr (UNIT == MT_CLAMPED)
        by = __builtin_bit_cast(float, number(next_tokens + ((1 + flip) * MT + p) * 4));
#pragma unroll
      for (int i = 0; i < 8; i += GLU ? 4 : 2) {
        float v[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if (GLU) {
              float z = sum(i + 2 * h, j, r), u = sum(i + 2 * h + 1, j, r);
              if constexpr (UNIT == MT_CLAMPED) {
                z = fminf(z * by, a.limit);
                u = fminf(fmaxf(u * by, -a.limit), a.limit) + 1.0f;
                v[h][r] = z * __builtin_amdgcn_rcpf(1.0f + __expf(-a.alpha * z)) * u;
              } else if constexpr (UNIT == MT_GELU) {
                // x (1 + tanh y) / 2 as x / (1 + exp(-2 y))
                const float y = 1.5957691216057308f * (z + 0.044715f * z * z * z);
                v[h][r] = z * __builtin_amdgcn_rcpf(1.0f + __expf(-y)) * u;
              } else {
                v[h][r] = z * __builtin_amdgcn_rcpf(1.0f + __expf(-z)) * u;
              }
            } else v[h][r] = sum(i + h, j, r);
          }
        // rows behind the last pair repeat it
        store(row, it.n0 + wn * (NC / 2) + i * (GLU ? 8 : 16), v[0], v[1]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    }
    lax = !PARTS && it.n0 + NC <= a.O ? 2 * R - 2 : 0;  // else some were left out
    it = nx;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#endif
}

// the stages that an item of MT pairs and K columns has room for
template <int MT, MoeUnit UNIT, int R, bool DENSE>
static void moe_tiles_launch(MoeTilesArgs& a, hipStream_t stream) {
  const bool gated = UNIT != MT_SUMS && UNIT != MT_PARTS;
  const int smem = R * (256 + MT) * 128 +
                   MT * 4 * (DENSE || !gated ? 0 : UNIT == MT_CLAMPED ? 3 : 1);
  (void)hipFuncSetAttribute(
      reinterpret_cast<const void*>(&moe_tiles_kernel<MT, UNIT, R, DENSE>),
      hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  const int across = gated ? 128 : 256;
  a.cols = (a.O + across - 1) / across;
  moe_tiles_kernel<MT, UNIT, R, DENSE><<<dim3(256), dim3(256), smem, stream>>>(a);
}

template <int MT, MoeUnit UNIT, bool DENSE = false>
static void moe_tiles_go(MoeTilesArgs& a, hipStream_t stream) {
  if (!DENSE) a.ldw = a.K * 2;
  if constexpr (MT == 256) {
    moe_tiles_launch<MT, UNIT, 2, DENSE>(a, stream);
  } else {
    // of two stages (K of 128) an item is shorter than three places
    if (DENSE || a.K > 128) moe_tiles_launch<MT, UNIT, 3, DENSE>(a, stream);
    else if constexpr (!DENSE) moe_tiles_launch<MT, UNIT, 2, DENSE>(a, stream);
  }
}
