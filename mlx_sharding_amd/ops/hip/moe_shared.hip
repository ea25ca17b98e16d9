// What stands before and behind the routed experts of a decoding step (moe_rows.hip), each
// together with half of the shared feed-forward, up to 64 tokens:
//
//   moe_begin   RMS norm, router product, softmax and choice of a token; beside them, on blocks
//               of their own, the shared units act(gate) * up of the normed rows
//   moe_finish  the shared units' product, which takes a token's weighted pairs and the residual
//               along
//
// A router is a chain of loads, sums and numbers that pass the L2s, during which the chip
// stands still (9.2 us of 64 tokens); the units, 10.4 us in a launch of their own, are read
// meanwhile, and both take 11.8, in one round of blocks.  The product takes 9.7 us with the
// pairs, 7.7 without them and 4.7 for their sum behind it.  64 experts of 1408 x 2048, 4 bits,
// 2816 shared units, a layer's feed-forward of 64 tokens 104 us, 94 so; of one, whose shared
// tiles went with the experts', 32.7 and 30.4.  Over 73 random layers of 9 to 64 tokens .86 of the
// time of the kernels apart; of 1 to 8 tokens up to 1.11 of that with the shared tiles among the
// experts' where rows are short and the matrices small, which stay there.  The router's blocks
// take 8 tokens: with one each, its blocks and those of the units, which have LDS for one of them
// a CU, are two rounds.
#include "linear_own_kernel.h"
#include "moe_rows.h"
#include "moe_choice.h"

namespace {

constexpr int ROUTED = 8;  // tokens of a router's block, a wave each

struct BeginArgs {
  LinearFewArgs units;
  MoeRouteArgs route;
  int N, parts, blocks;  // parts: of 16 experts; blocks: of the router, a multiple of 8
};

// Columns of a row in the router's LDS: a row is off the next one's banks by 16 bytes.
__host__ __device__ constexpr int routed_row(int H) { return H + 8; }

// 8 tokens by 16 experts; the wave that has a token's last logits chooses for it.
__device__ __forceinline__ void route_block(const BeginArgs& b) {
  const MoeRouteArgs& a = b.route;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __bf16* rows = reinterpret_cast<__bf16*>(smem);
  __shared__ float part[OWN_WAVES][WAVE * 4];
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int l16 = lane & 15, lg = lane >> 4;
  const int group = blockIdx.x / b.parts, first = (blockIdx.x - group * b.parts) * 16;
  const int t0 = group * ROUTED, n = min(ROUTED, b.N - t0);
  if (n <= 0) return;
  const int ld = routed_row(a.H);
  auto load = [](const __bf16* p) { return *reinterpret_cast<const bf16x8_t*>(p); };

  // this wave's row, up to 4096 columns of it
  constexpr int PIECES = 8;
  bf16x8_t v[PIECES], g[PIECES];
  const long t = t0 + wid;
  if (wid < n) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int col = (i * WAVE + lane) * 8;
      if (col >= a.H) continue;
      v[i] = load(a.x + t * a.H + col);
      g[i] = load(a.norm + col);
    }
  }
  // its eighth of the contraction, in steps of 32
  const int steps = a.H / 32, per = (steps + OWN_WAVES - 1) / OWN_WAVES;
  const int s0 = wid * per, s1 = min(steps, s0 + per);
  const __bf16* from = a.gate + (long)min(first + l16, a.E - 1) * a.H + lg * 8;
  constexpr int HELD = 8;
  bf16x8_t w[HELD];
#pragma unroll
  for (int i = 0; i < HELD; ++i) w[i] = load(from + min(s0 + i, steps - 1) * 32);

  if (wid < n) {
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      if ((i * WAVE + lane) * 8 >= a.H) continue;
#pragma unroll
      for (int j = 0; j < 8; ++j) ss = fmaf((float)v[i][j], (float)v[i][j], ss);
    }
    const float f = rsqrtf(wave_sum(ss) / a.H + a.eps);
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int col = (i * WAVE + lane) * 8;
      if (col >= a.H) continue;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        v[i][j] = (__bf16)((float)v[i][j] * f * ((float)g[i][j] + a.offset));
      *reinterpret_cast<bf16x8_t*>(rows + wid * ld + col) = v[i];
      if (first == 0) *reinterpret_cast<bf16x8_t*>(a.y + t * a.H + col) = v[i];
    }
  }
  __syncthreads();
  const __bf16* x = rows + min(l16, n - 1) * ld + lg * 8;
  f32x4 acc[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
  for (int s = s0; s < s1; s += HELD) {
#pragma unroll
    for (int i = 0; i < HELD; ++i)
      if (s + i < s1)
        acc[i & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i], load(x + (s + i) * 32),
                                                             acc[i & 1], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < HELD; ++i)
      if (s + HELD + i < s1) w[i] = load(from + (s + HELD + i) * 32);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) part[wid][lane * 4 + j] = acc[0][j] + acc[1][j];
  __syncthreads();
  if (wid >= n) return;
  // lane: an expert; its sums lie with the token's lanes
  float z = 0.0f;
#pragma unroll
  for (int p = 0; p < OWN_WAVES; ++p)
    z += part[p][((l16 >> 2) * 16 + wid) * 4 + (l16 & 3)];
  float* logits = a.logits + t * 64;
  if (lane < 16)
    __hip_atomic_store(logits + first + lane, z, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  unsigned before = 0;
  if (lane == 0)
    before = __hip_atomic_fetch_add(a.tickets + t, 1u, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT);
  if (__builtin_amdgcn_readfirstlane(before) + 1 != (unsigned)b.parts) return;
  asm volatile("" ::: "memory");
  z = lane < a.E ? __hip_atomic_load(logits + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                 : -INFINITY;
  int place;
  float weight;
  if (chosen_expert(z, lane, a.E, a.top, a.normalize, a.scaling, place, weight)) {
    a.choice[t * a.top + place] = lane;
    a.weight[t * a.top + place] = weight;
  }
}

template <int RT, int TT>
__global__ __launch_bounds__(OWN_WAVES * WAVE) void moe_begin_kernel(const BeginArgs b) {
  if ((int)blockIdx.x < b.blocks) route_block(b);
  else own_block<RT, TT, 1, true, true, false, false>(b.units, blockIdx.x - b.blocks);
}

template <int RT, int TT>
__global__ __launch_bounds__(OWN_WAVES * WAVE) void moe_finish_kernel(const LinearFewArgs a) {
  own_block<RT, TT, RT == 1 ? 2 : 1, false, false, false, true>(a, blockIdx.x);
}

template <typename Kernel, typename Args>
void go(Kernel kernel, const Args& a, int blocks, int smem, hipStream_t stream) {
  if (smem > 48 * 1024)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  kernel<<<blocks, OWN_WAVES * WAVE, smem, stream>>>(a);
}

}  // namespace

// w_in [2 S, H], units [N, S]
extern "C" void launch_moe_begin(const MoeRouteArgs* r, int N, const void* w_in, void* units,
                                 int S, hipStream_t stream) {
  BeginArgs b{};
  b.route = *r;
  b.N = N;
  b.parts = (r->E + 15) / 16;
  b.blocks = ((N + ROUTED - 1) / ROUTED * b.parts + 7) / 8 * 8;
  LinearFewArgs& a = b.units;
  a.x = r->x, a.w = (const __bf16*)w_in, a.norm = r->norm, a.y = (__bf16*)units;
  a.M = (short)N, a.O = S, a.K = r->H;
  a.ldx = a.ldw = r->H, a.ldy = S;
  a.eps = r->eps, a.offset = r->offset;
  turned(a, LF_SILU, 64);
  const Tiles t = tiles_beside(N, (S + 7) / 8, b.blocks, r->H, true);
  const int rows = ROUTED * routed_row(r->H) * 2;
  with_tiles(t, [&](auto rt, auto tt) {
    go(&moe_begin_kernel<rt(), tt()>, b, b.blocks + t.blocks,
       max(rows, own_room(t.rt, t.tt, 1, a.K, true)), stream);
  });
}

// units [N, S], w_out [H, S], rows [N * top, H], h and out [N, H]
extern "C" void launch_moe_finish(const void* units, const void* w_out, const float* rows,
                                  const void* h, void* out, int N, int H, int S, int top,
                                  hipStream_t stream) {
  LinearFewArgs a{};
  a.x = (const __bf16*)units, a.w = (const __bf16*)w_out, a.res = (const __bf16*)h;
  a.y = (__bf16*)out, a.part = const_cast<float*>(rows);
  a.M = (short)N, a.O = H, a.K = S, a.n_zero = top;
  a.ldx = a.ldw = S, a.ldr = a.ldy = H;
  a.fours = 1;
  turned(a, LF_PLAIN, 64);
  const Tiles t = tiles_beside(N, H / 16, 0, S, false);
  with_tiles(t, [&](auto rt, auto tt) {
    go(&moe_finish_kernel<rt(), tt()>, a, t.blocks,
       own_room(t.rt, t.tt, t.rt == 1 ? 2 : 1, S, false), stream);
  });
}
