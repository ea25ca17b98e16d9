// Products of routed experts over tiles of one expert's (token, expert) pairs.
//
// What bounds them: the matrix cores.  A block of four waves makes 256 pairs
// by 256 rows of weights, a wave 128 x 128, whose sums fill the accumulation
// registers: a step of 32 columns then takes 1024 cycles of every core and half as
// many of LDS.  Four stages of LDS are a ring: while one is worked on, the next is
// complete and two are on their way, straight from memory.  Operands of a half step
// are read and loads are asked for between the products of the half step before; one
// barrier a step.  A block walks over its tiles without a gap: behind a tile's last
// stage the ring goes on with the next one's, and results are stored meanwhile.
// Pieces of 16 bytes within a row of 64 are swapped by the row, so that rows that a
// read meets lie in different banks.
// Measured: 32768 tokens, top 6 of 64 experts, 2048 -> 1408: 1.94 ms (1167 TFLOP/s),
// 1408 -> 2048: 1.15 (984); with a block per tile 2.07 and 1.29, loads in one run
// behind the barrier 2.31 and 1.39.
// Clamped units read their pairs' weights out of LDS at the end of an item, where a load
// from memory would wait for the stages under way.
#pragma once

#include "moe_tiles.h"

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

#define MT_GROUP 4  // tiles whose blocks run together, with the same weights
// MT: pairs of a tile
template <int MT, MoeUnit UNIT>
__global__ __launch_bounds__(256, 1) void moe_tiles_kernel(const MoeTilesArgs a) {
  constexpr bool GLU = UNIT != MT_SUMS;
  constexpr int NP = MT / 64;          // 32-pair tiles of a wave
  constexpr int L = 4 + NP;            // loads per wave and stage
  constexpr int ST = (256 + MT) * 64;  // bytes of a stage
  constexpr int NC = GLU ? 128 : 256;  // outputs of a block
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, hi = lane >> 5;
  const int wm = wid >> 1, wn = wid & 1;
  const int nk = a.K / 32;

  // an XCD has consecutive tiles, its blocks walk them in groups
  const int total = *a.n_tiles;
  const int group = total >= 16 * MT_GROUP ? MT_GROUP : 1;  // few: to all XCDs
  const int per = (total + 8 * group - 1) / (8 * group) * group;
  const int xcd = blockIdx.x & 7, step = gridDim.x >> 3;
  int slot = (int)(blockIdx.x >> 3) - step;
  struct Item { int e, p0, np, n0; };
  struct Place { int tile, n0; };  // a tile, or -1 behind the last one
  auto advance = [&]() -> Place {
    for (;;) {
      slot += step;
      const int grp = slot / (group * a.cols), rest = slot % (group * a.cols);
      const int ti = grp * group + rest % group;
      if (ti >= per) return {-1, 0};
      if (xcd * per + ti < total) return {xcd * per + ti, rest / group * NC};
    }
  };
  // a tile's entry is asked for an item ahead, by vector loads: one that is waited
  // for where it is needed would wait for all that was stored before it
  int nought = 0;
  asm volatile("" : "+v"(nought));
  struct Entry { int e, p0, np; };
  auto entry = [&](int tile) -> Entry {
    const int* t = a.tiles + max(tile, 0) * 3 + nought;
    return {t[0], t[1], t[2]};
  };
  auto item = [&](const Entry& x, int n0) -> Item {
    return {__builtin_amdgcn_readfirstlane(x.e), __builtin_amdgcn_readfirstlane(x.p0),
            __builtin_amdgcn_readfirstlane(x.np), n0};
  };
  auto place = [](int row, int piece) { return piece ^ ((row >> 2) & 3); };
  // A wave's rows of a stage: bases that it shares, 32-bit offsets from there.  Of a
  // gated unit, waves 0 and 1 bring gate rows, 2 and 3 up rows (32 by turns).
  struct Rows { const char *w, *x; unsigned off[L]; };
  auto tokens = [&](const Item& it, int (&t)[NP]) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int p = min((i * 4 + wid) * 16 + (lane >> 2), it.np - 1);
      t[i] = GLU ? a.tokens[it.p0 + p] : p;
    }
  };
  auto rows_of = [&](const Item& it, const int (&t)[NP], Rows& s) {
    s.w = (GLU && wid >> 1 ? a.w2 : a.w) + it.e * a.wstride;
    s.x = a.x + (GLU ? 0 : it.p0 * a.xstride);
#pragma unroll
    for (int i = 0; i < L; ++i) {
      const int r = (i % 4 * 4 + wid) * 16 + (lane >> 2);
      const int piece = place(r, lane & 3);
      if (i < 4) {
        const int o = it.n0 + (GLU ? (r >> 7) * 64 + (r >> 6 & 1) * 32 + (r & 31) : r);
        s.off[i] = (unsigned)min(o, a.O - 1) * (unsigned)(a.K * 2) + piece * 16;
      } else {
        s.off[i] = (unsigned)t[i - 4] * (unsigned)a.xstride + piece * 16;
      }
    }
  };
  auto load = [&](const Rows& s, int k, int g, int i) {
    const int part = i < 4 ? i * 4 + wid : 16 + (i - 4) * 4 + wid;
    const char* base = (i < 4 ? s.w : s.x) + k * 64;
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) void*)(base + s.off[i]),
        (__attribute__((address_space(3))) void*)(smem + (g & 3) * ST + part * 1024), 16, 0, 0);
  };
  Place at = advance();
  if (at.tile < 0) return;
  Item it = item(entry(at.tile), at.n0);
  at = advance();
  Entry ahead = entry(at.tile);
  int tok[NP];
  Rows rows;
  tokens(it, tok);
  rows_of(it, tok, rows);

  f32x16 acc[4][NP];
  struct Frags { bf16x8_t w[4], x[NP]; };
  int wo[2], xo[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int pl = place(l32, 2 * s + hi) * 16;
    wo[s] = (wn * 128 + l32) * 64 + pl;
    xo[s] = (256 + wm * (MT / 2) + l32) * 64 + pl;
  }
  auto rd = [](const char* p) { return *reinterpret_cast<const bf16x8_t*>(p); };
  // products of `f`; between them operands of the next half step and loads
  auto half = [&](const Frags& f, Frags& n, int g, int s, auto&& fetch) {
    const char* b = smem + (g & 3) * ST;
    auto wr = [&](int i) { n.w[i] = rd(b + wo[s] + i * 2048); };
    auto xr = [&](int i) { if (i < NP) n.x[i] = rd(b + xo[s] + i * 2048); };
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int j = 0; j < NP; ++j) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.w[i], f.x[j], acc[i][j], 0, 0, 0);
        if (j == 0) {
          __builtin_amdgcn_sched_barrier(0);
          if (i == 0) { wr(0); xr(0); xr(1); }
          if (i == 1) { wr(1); xr(2); xr(3); }
          if (i == 2) { wr(2); wr(3); }
          fetch(i);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int g = 0; g < 3; ++g)
#pragma unroll
    for (int i = 0; i < (g < 2 ? L : L / 2); ++i) load(rows, g, g, i);
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"(L + L / 2) : "memory");
  __builtin_amdgcn_sched_barrier(0);
  Frags f0, f1;
#pragma unroll
  for (int i = 0; i < 4; ++i) f0.w[i] = rd(smem + wo[0] + i * 2048);
#pragma unroll
  for (int i = 0; i < NP; ++i) f0.x[i] = rd(smem + xo[0] + i * 2048);

  int g = 0;  // stages so far
  int flip = 0;
  for (bool more = true; more;) {
    more = at.tile >= 0;
    const Item nx = more ? item(ahead, at.n0) : it;
    if (more) at = advance();
    ahead = entry(at.tile);
    tokens(nx, tok);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < NP; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    // weights of this item's pairs go to LDS, and are there some steps later; those of
    // the item before may still be read
    if constexpr (UNIT == MT_CLAMPED) {
      flip ^= 1;
      if (wid * 64 < MT)
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void*)(
                a.scale + it.p0 + min(wid * 64 + lane, it.np - 1)),
            (__attribute__((address_space(3))) void*)(
                smem + 4 * ST + (flip * MT + wid * 64) * 4), 4, 0, 0);
    }
    auto step = [&](auto&& fetch) {
      half(f0, f1, g, 1, [&](int i) {
        if (L / 2 + i < L) fetch(2, L / 2 + i);
      });
      __builtin_amdgcn_s_waitcnt(0x70 | L);
      asm volatile("s_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      half(f1, f0, g + 1, 0, [&](int i) {
        if (i < L / 2) fetch(3, i);
      });
    };
    int k = 0;
    do {  // 4 stages at least
      step([&](int d, int i) { load(rows, k + d, g + d, i); });
      ++k, ++g;
    } while (k < nk - 3);
    // behind the last stage of this item come the next one's
    Rows next;
    rows_of(nx, tok, next);
    for (; k < nk; ++k, ++g)
      step([&](int d, int i) {
        const bool same = k + d < nk;
        load(same ? rows : next, same ? k + d : k + d - nk, g + d, i);
      });
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
    // lane: pair l32, outputs (r & 3) + 8 (r >> 2) + 4 hi of 32
    auto store = [&](__bf16* row, int o, const float (&lo)[4], const float (&up)[4]) {
      u32x2 x, y;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        x[h] = __builtin_bit_cast(unsigned, bf16x2_t{(__bf16)lo[2 * h], (__bf16)lo[2 * h + 1]});
        y[h] = __builtin_bit_cast(unsigned, bf16x2_t{(__bf16)up[2 * h], (__bf16)up[2 * h + 1]});
      }
      const auto s0 = __builtin_amdgcn_permlane32_swap(x[0], y[0], false, false);
      const auto s1 = __builtin_amdgcn_permlane32_swap(x[1], y[1], false, false);
      o += hi * 8;
      if (o < a.O) *reinterpret_cast<u32x4*>(row + o) = u32x4{s0[0], s1[0], s0[1], s1[1]};
    };
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      const int p = wm * (MT / 2) + j * 32 + l32;
      // all lanes take part in the exchange
      __bf16* row = a.y + (long)(it.p0 + min(p, it.np - 1)) * a.O;
      // read here: the compiler would wait for all loads to LDS
      float by = 1.0f;
      if constexpr (UNIT == MT_CLAMPED) {
        const auto* at = (__attribute__((address_space(3))) char*)(
            smem + 4 * ST + (flip * MT + p) * 4);
        asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(by) : "v"(at) : "memory");
      }
#pragma unroll
      for (int i = 0; i < (GLU ? 2 : 4); ++i)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          float v[2][4];
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int c = (2 * q + h) * 4 + r;
              if (GLU) {
                float z = sum(2 * i, j, c), u = sum(2 * i + 1, j, c);
                if constexpr (UNIT == MT_CLAMPED) {
                  z = fminf(z * by, a.limit);
                  u = fminf(fmaxf(u * by, -a.limit), a.limit) + 1.0f;
                  v[h][r] = z * __builtin_amdgcn_rcpf(1.0f + __expf(-a.alpha * z)) * u;
                } else {
                  v[h][r] = z * __builtin_amdgcn_rcpf(1.0f + __expf(-z)) * u;
                }
              } else v[h][r] = sum(i, j, c);
            }
          const int o = it.n0 + wn * (NC / 2) + i * 32 + q * 16;
          // rows behind the last pair repeat it
          store(row, o, v[0], v[1]);
          __builtin_amdgcn_sched_barrier(0);
        }
    }
    it = nx;
    rows = next;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

template <int MT, MoeUnit UNIT>
static void moe_tiles_go(MoeTilesArgs& a, hipStream_t stream) {
  const int smem = 4 * (256 + MT) * 64 + (UNIT == MT_CLAMPED ? 2 * MT * 4 : 0);
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&moe_tiles_kernel<MT, UNIT>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  const int across = UNIT != MT_SUMS ? 128 : 256;
  a.cols = (a.O + across - 1) / across;
  moe_tiles_kernel<MT, UNIT><<<dim3(256), dim3(256), smem, stream>>>(a);
}
