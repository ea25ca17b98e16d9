// Causal attention of a prompt on matrix cores (mfma_f32_32x32x16_bf16).
//
// A wave owns 32 queries of one head.  Scores are computed transposed, S^T = K
// Q^T, so that a lane holds scores of one query only: softmax needs one exchange
// between the two halves of the wave, and the weights, rounded to bf16, are the
// second product's operand (O^T = V^T P^T) without leaving their lanes.
//
//   mfma_f32_32x32x16_bf16: A (32x16) lane: row l&31, contraction (l>>5)*8 + j
//                           B (16x32) lane: col l&31, contraction (l>>5)*8 + j
//                           C (32x32) lane: col l&31, reg r is row
//                                     (r&3) + 8*(r>>2) + 4*(l>>5)
//
// The order of contraction indices is free as long as A and B agree, so V^T is
// read in the order in which a lane's scores lie: two groups of four keys.
// ds_read_b64_tr_b16 gives a lane four keys of one column out of rows of V, so V
// lies in LDS as it lies in memory.
//
// What bounds it: the matrix cores and the exponentials and maxima between them,
// which alternate in one wave; two waves a SIMD fill each other's gaps, the one that
// multiplies first (s_setprio: 8192 tokens as below 534 -> 525 us, of 256 behind 4096
// 208 -> 190).  Tiles of 64 keys have the exponentials among the second products, which a
// wave alone on its SIMD needs (2048 tokens: 55 us with the priority raised between, 50.5
// so, 52.2 before); tiles of 32 of 256 columns have no registers for that (215 us, 190).
// Keys and values of a tile go to LDS without passing registers, the next tile while
// this one is worked on (that the compiler has the reads of values wait for it costs
// nothing: without 559.8 us, 559.7).  16-byte pieces of a row are swapped by the row's low bits
// (on their way from memory, the place in LDS is fixed), without which the rows
// that a read meets share their banks.
// Measured (before: 16 queries a wave, scores through LDS, V transposed element by
// element): 8192 tokens, 32 heads of 128 over 8: 5310 -> 525 us (1047 TFLOP/s);
// 4096 tokens, 16 heads of 256 over 8, capped: 1600 -> 173 us (794), 1905 behind 4096
// with a window of 4096: 161 us (400 and 450 while places in LDS had a register each
// and were spilled: each reload waited for the next tile's loads; 13 and 15 us more with
// all of a query in registers); 64 prompts of 512, 16 heads of 192/128: 1216 -> 176 us
// (490); 57 tokens: 8.4 -> 7.6 us.

#include <algorithm>

#include "hip_common.h"
#include "soft_cap.h"

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

#define AP_WAVES 4
#define AP_BLOCK (AP_WAVES * WAVE)

struct PrefillArgs {
  const char *q, *k, *v;
  char* out;
  int Hq, Hkv, T, S;
  long q_b, q_h, q_t;        // strides of q, elements
  long kcap, vcap;           // rows of a head's keys and values
  float c;                   // score -> power of two; behind a cap: 1
  SoftCap cap;
  int flip;                  // a negative scale: queries change their sign
  int window, offset;
  int heads, tiles, group;   // B * Hq, query tiles, heads that run together
  // keys in two parts (latent attention): k and v are columns of rows [B, S, Hq,
  // NOPE + DV], a key's last DK - NOPE columns are a row of `pe` for all heads;
  // queries turn by their positions
  const char* pe;
  long pe_b;                 // bytes from one sequence to the next
  int kv_row, pe_row;        // bytes from one key to the next
  const float *cos, *sin;    // [T, (DK - NOPE) / 2]
  // portions of a batch, rows of queries and of keys one behind the other; keys'
  // first columns and values in rows of their own, queries have been turned
  const int *portions;       // [tiles, 2]: request, first row
  const int *cu, *pos0, *cuk;
  int n_short, tok_base, v_row;
};

// 16 bytes a lane from memory to LDS, lane after lane from `dst` on
__device__ __forceinline__ void ap_to_lds(const char* src, char* dst) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) void*)src,
      (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

// the larger of a lane's value and that of its partner in the other half
__device__ __forceinline__ float other_half_max(float x) {
  const unsigned u = __float_as_uint(x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// Place of a 16-byte piece within its row in LDS: keys are read a row a lane,
// values four rows by 32 bytes a quarter wave.
template <int N>
__device__ __forceinline__ int key_place(int row, int piece) {
  return N >= 8 ? piece ^ (row & 7) : piece ^ ((row >> 1) & 3);
}
template <int N>
__device__ __forceinline__ int value_place(int row, int piece) {
  if (N >= 16) return piece ^ ((row & 7) << 1);
  if (N == 8) return piece ^ ((row & 3) << 1);
  if (N == 4) return piece ^ ((row >> 1 & 1) << 1);
  return piece;
}

// keys of a tile
constexpr int ap_keys(int DK, int DV) { return DK + DV > 320 ? 32 : 64; }

// NOPE: columns of a key that lie with the values, 0: rows of keys and of values.
// RAGGED: portions of a batch; weights enter the second product in two bf16 parts, as
// they do in that cache's other kernels.
// TEAMS: of four waves each, with tiles of their own, that share the keys of the same
// queries by turns and add up through LDS.
template <int DK, int DV, bool CAP, int TEAMS, int NOPE = 0, bool RAGGED = false>
__global__ __launch_bounds__(AP_BLOCK* TEAMS, 2) void attn_prefill_kernel(
    const PrefillArgs a) {
  constexpr int KT = ap_keys(DK, DV);
  constexpr int KP = DK / 8, VP = DV / 8;      // pieces of a row
  constexpr int NK = DK / 16, NB = KT / 32, ND = (DV + 31) / 32;
  constexpr int KB = KT * DK * 2, VB = KT * DV * 2;
  // The last pieces of queries of 256 lie in LDS: they and the sums leave too few
  // registers to read keys and values ahead of their products.
  constexpr int QL = DK == 256 ? 4 : 0;
  // a lane of the columns behind DV = 16 reads past its row
  constexpr int OWN = 2 * (KB + VB) + AP_WAVES * QL * 1024 + (DV < 32 ? 64 : 0);
  __shared__ __attribute__((aligned(16))) char smem_all[TEAMS * OWN];

  // Blocks go round the XCDs.  Each XCD takes whole heads, `group` of them at a
  // time, and their longest tiles first: heads that share keys share an L2.
  int head, tile;
  if (a.heads % 8 == 0) {
    const int slot = blockIdx.x >> 3, run = a.group * a.tiles;
    head = (blockIdx.x & 7) * (a.heads >> 3) + slot / run * a.group +
           slot % run % a.group;
    tile = a.tiles - 1 - slot % run / a.group;
  } else {
    head = blockIdx.x % a.heads;
    tile = a.tiles - 1 - blockIdx.x / a.heads;
  }
  const int b = head / a.Hq, h = head % a.Hq;
  const long kv = (long)b * a.Hkv + h / (a.Hq / a.Hkv);
  int q0 = tile * (AP_WAVES * 32), T = a.T, S = a.S, offset = a.offset;
  long t0 = 0, k0 = 0;
  if (RAGGED) {
    const int e = a.portions[2 * tile];
    q0 = a.portions[2 * tile + 1];
    t0 = a.cu[e];
    T = a.cu[e + 1] - (int)t0;
    offset = a.pos0[e];
    S = offset + T;
    k0 = a.cuk[e - a.n_short];
  }
  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int team = wave / AP_WAVES, wid = wave % AP_WAVES;
  char* smem = smem_all + team * OWN;
  const int l32 = lane & 31, hi = lane >> 5;
  const char *kbase, *vbase, *pbase = nullptr;
  if (RAGGED) {
    kbase = a.k + k0 * a.kv_row + (long)h * NOPE * 2;
    vbase = a.v + k0 * a.v_row + (long)h * DV * 2;
    pbase = a.pe + k0 * a.pe_row;
  } else if (NOPE) {
    kbase = a.k + (long)b * a.S * a.kv_row + (long)h * (NOPE + DV) * 2;
    vbase = kbase + NOPE * 2;
    pbase = a.pe + (long)b * a.pe_b;
  } else {
    kbase = a.k + kv * a.kcap * (DK * 2);
    vbase = a.v + kv * a.vcap * (DV * 2);
  }
  const int krow_w = NOPE ? a.kv_row : DK * 2, vrow_w = RAGGED ? a.v_row : NOPE ? a.kv_row : DV * 2;

  // rows behind the last key repeat it; their weights are zero
  auto stage = [&](int t, int buf) {
    char* dst = smem + buf * (KB + VB);
    const char* ks = kbase + (long)t * krow_w;
    const char* vs = vbase + (long)t * vrow_w;
    const char* ps = NOPE ? pbase + (long)t * a.pe_row : nullptr;
    const int last = S - 1 - t;
#pragma unroll
    for (int i = 0; i < KB / 1024; i += AP_WAVES) {
      const int part = i + wid;
      if (KB / 1024 % AP_WAVES && part >= KB / 1024) break;
      const int s = part * 64 + lane, row = s / KP;
      const int piece = key_place<KP>(row, s % KP);
      const char* src = ks + min(row, last) * krow_w + piece * 16;
      if (NOPE && piece >= NOPE / 8)
        src = ps + min(row, last) * a.pe_row + (piece - NOPE / 8) * 16;
      ap_to_lds(src, dst + part * 1024);
    }
#pragma unroll
    for (int i = 0; i < VB / 1024; i += AP_WAVES) {
      const int part = i + wid;
      if (VB / 1024 % AP_WAVES && part >= VB / 1024) break;
      const int s = part * 64 + lane, row = s / VP;
      ap_to_lds(vs + min(row, last) * vrow_w +
                    value_place<VP>(row, s % VP) * 16, dst + KB + part * 1024);
    }
  };

  const int end = min(S, offset + min(q0 + AP_WAVES * 32, T));
  int from = 0;
  if (a.window > 0) from = max(0, offset + q0 - a.window + 1) & ~(KT - 1);
  constexpr int TURN = TEAMS * KT;
  const int turns = (max(end - from, 0) + TURN - 1) / TURN;
  from += team * KT;
  if (from < end) stage(from, 0);

  const int w0 = q0 + wid * 32;  // this wave's first query
  const int row = min(w0 + l32, T - 1);
  const int qpos = min(offset + row, S - 1);       // last key seen
  const int qfrom = a.window > 0 ? offset + row - a.window + 1 : 0;
  bf16x8_t qf[NK];
  char* ql = smem + 2 * (KB + VB) + (wid * QL * WAVE + lane) * 16;
  {
    const char* src =
        a.q + ((long)b * a.q_b + (long)h * a.q_h + (t0 + row) * a.q_t) * 2 + hi * 16;
#pragma unroll
    for (int i = 0; i < NK; ++i)
      qf[i] = *reinterpret_cast<const bf16x8_t*>(src + i * 32);
    if (NOPE && !RAGGED) {
      // as rounded rows of queries would be
#pragma unroll
      for (int i = NOPE / 16; i < NK; ++i) {
        const long at = (long)row * ((DK - NOPE) / 2) + (i * 16 + hi * 8 - NOPE) / 2;
        const f32x4 c = *reinterpret_cast<const f32x4*>(a.cos + at);
        const f32x4 n = *reinterpret_cast<const f32x4*>(a.sin + at);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float x = (float)qf[i][2 * j], y = (float)qf[i][2 * j + 1];
          qf[i][2 * j] = (__bf16)(x * c[j] - y * n[j]);
          qf[i][2 * j + 1] = (__bf16)(y * c[j] + x * n[j]);
        }
      }
    }
    if (a.flip) {
#pragma unroll
      for (int i = 0; i < NK; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) qf[i][j] = -qf[i][j];
    }
  }
#pragma unroll
  for (int i = 0; i < QL; ++i)
    *reinterpret_cast<bf16x8_t*>(ql + i * 1024) = qf[NK - QL + i];
  // keys that all of the wave's queries see, and those that any of them sees
  const int all_hi = min(offset + min(w0, T - 1), S - 1);
  const int any_hi = w0 < T ? min(offset + min(w0 + 31, T - 1), S - 1) : -1;
  const int all_lo = a.window > 0 ? offset + min(w0 + 31, T - 1) - a.window + 1 : 0;
  const int any_lo = a.window > 0 ? offset + w0 - a.window + 1 : 0;

  float m = -1e30f, l = 0.0f;  // reference of the exponents (base 2), sum
  f32x16 o[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.0f;

  const int krow = l32 * KP * 16;
  const int i16 = lane & 15;
  const int vkey = hi * 4 + (i16 >> 2);
  // Swapping moves a piece within 8 of keys, 16 of values: four places, the others lie
  // behind them.
  int kplace[NK < 4 ? NK : 4], vplace[ND < 4 ? ND : 4];
#pragma unroll
  for (int i = 0; i < (NK < 4 ? NK : 4); ++i)
    kplace[i] = krow + key_place<KP>(l32, 2 * i + hi) * 16;
#pragma unroll
  for (int d = 0; d < (ND < 4 ? ND : 4); ++d)
    vplace[d] = vkey * VP * 16 + (i16 & 1) * 8 +
                value_place<VP>(vkey, d * 4 + (lane >> 4 & 1) * 2 + (i16 >> 1 & 1)) * 16;
  auto work = [&](int t, auto which) {
    constexpr int buf = decltype(which)::value;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t + TURN < end) stage(t + TURN, buf ^ 1);
    if (t > any_hi || t + KT <= any_lo) return;
    const char* kt = smem + buf * (KB + VB);
    const char* vt = kt + KB;

    __builtin_amdgcn_s_setprio(1);
    f32x16 s[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[n][r] = 0.0f;
#pragma unroll
    for (int i = 0; i < NK; ++i)
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        const bf16x8_t f = *reinterpret_cast<const bf16x8_t*>(
            kt + n * 32 * KP * 16 + i / 4 * 128 + kplace[i % 4]);
        const bf16x8_t q = i < NK - QL ? qf[i] : *reinterpret_cast<const bf16x8_t*>(
                                                     ql + (i - NK + QL) * 1024);
        s[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f, q, s[n], 0, 0, 0);
      }
    // three of the tile's reads before the first product, then one a product: what the
    // compiler arranges waits for every second read
    constexpr int READS = NK * NB, AHEAD = READS < 3 ? READS : 3;
    __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
    for (int i = 0; i < READS - AHEAD; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, AHEAD, 0);
    __builtin_amdgcn_s_setprio(0);
    if (CAP) {
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        float v[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r] = s[n][r];
        soft_capped(a.cap, v);
#pragma unroll
        for (int r = 0; r < 16; ++r) s[n][r] = v[r];
      }
    }
    if (t + KT - 1 > all_hi || t < all_lo) {
#pragma unroll
      for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = t + n * 32 + (r & 3) + 8 * (r >> 2) + 4 * hi;
          if (key > qpos || key < qfrom) s[n][r] = -INFINITY;
          // four at a time: of more, masks go to other registers and back (one prompt
          // of 8 heads of 64, capped, 512 tokens: 16.1 us, 14.9 so)
          if (CAP && r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
    }
    float top = -INFINITY;
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) top = fmaxf(top, s[n][r]);
    top = other_half_max(top) * a.c;
    // The reference moves where a score is 2^8 above it: below that weights and
    // sums of a tile are as exact, and the outputs need not be scaled.
    if (__any(top > m + 8.0f)) {
      const float m_new = fmaxf(m, top);
      const float f = __builtin_amdgcn_exp2f(m - m_new);
      m = m_new;
      l *= f;
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] *= f;
    }
    float sum = 0.0f;
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[n][r] = __builtin_amdgcn_exp2f(fmaf(s[n][r], a.c, -m));
        sum += s[n][r];
      }
    l += sum;
    if (KT == 32) __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int x = 0; x < KT / 16; ++x) {
      bf16x8_t p, rest;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float w = s[x / 2][x % 2 * 8 + j];
        p[j] = (__bf16)w;
        if (RAGGED) rest[j] = (__bf16)(w - (float)p[j]);
      }
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        const char* src = vt + x * 16 * VP * 16 + d / 4 * 256 + vplace[d % 4];
        const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)src);
        const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(src + 8 * VP * 16));
        const short8v v = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            __builtin_bit_cast(bf16x8_t, v), p, o[d], 0, 0, 0);
        if (RAGGED)
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              __builtin_bit_cast(bf16x8_t, v), rest, o[d], 0, 0, 0);
      }
    }
  };
  // two of its tiles at a time: where a tile lies is known
  for (int i = 0; i < turns; i += 2) {
    work(from + i * TURN, std::integral_constant<int, 0>());
    if (i + 1 < turns) work(from + (i + 1) * TURN, std::integral_constant<int, 1>());
  }

  if constexpr (TEAMS == 2) {
    constexpr int EACH = ND * 16 + 2;
    static_assert(AP_WAVES * EACH * WAVE * 4 <= TEAMS * OWN, "sums fit");
    float* of = reinterpret_cast<float*>(smem_all) + wid * EACH * WAVE + lane;
    __syncthreads();  // all of the tiles are read
    if (team == 1) {
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) of[(d * 16 + r) * WAVE] = o[d][r];
      of[ND * 16 * WAVE] = m;
      of[(ND * 16 + 1) * WAVE] = l;
    }
    __syncthreads();
    if (team == 1) return;
    const float m2 = of[ND * 16 * WAVE], l2 = of[(ND * 16 + 1) * WAVE];
    const float top = fmaxf(m, m2);
    const float f1 = __builtin_amdgcn_exp2f(m - top), f2 = __builtin_amdgcn_exp2f(m2 - top);
    l = l * f1 + l2 * f2;
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        o[d][r] = o[d][r] * f1 + of[(d * 16 + r) * WAVE] * f2;
  }
  l += __shfl_xor(l, 32, WAVE);
  if (w0 + l32 >= T) return;
  const float f = 1.0f / l;
  // out [B, T, Hq, DV]
  const long at = RAGGED ? t0 - a.tok_base : (long)b * T;
  char* dst = a.out + (((at + w0 + l32) * a.Hq + h) * DV + hi * 4) * 2;
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (d * 32 + g * 8 >= DV) break;
      bf16x4_t w;
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = (__bf16)(o[d][g * 4 + j] * f);
      *reinterpret_cast<bf16x4_t*>(dst + (d * 32 + g * 8) * 2) = w;
    }
}

// head sizes (keys, values) that there is a kernel for
#define AP_SIZES(DO)                                                       \
  DO(32, 16) DO(32, 32) DO(32, 64) DO(64, 32) DO(64, 64) DO(64, 128)       \
  DO(128, 32) DO(128, 64) DO(128, 128) DO(192, 64) DO(192, 128) DO(256, 256)

// Callers must check this first: other sizes launch nothing.
extern "C" bool attn_prefill_supported(int Dk, int Dv) {
#define AP_HAS(K, V) if (Dk == K && Dv == V) return true;
  AP_SIZES(AP_HAS)
#undef AP_HAS
  return false;
}

// A block of one team leaves a SIMD one wave while it has a CU to itself: where there are
// no more blocks than CUs, and at the end of a causal prompt of two blocks a CU, which
// the longest blocks are alone with.  Two teams fill it and halve the chain of tiles;
// adding them up costs 1 to 2 us, so the chain has to be long, and blocks of like length
// gain nothing.  One team, two, us: 16 heads of 256, capped: 1905 tokens behind 4096 264,
// 206 (with a window of 4096 197, 161), 384 24.7, 24.5, 320 19.7, 20.6, 64 8.0, 10.5; 4096
// (512 blocks) 212, 173, with a window of 1024 95, 110; not capped 512 27.1, 26.8, 448 22.3,
// 22.6; 32 of 128: 1024 24.0, 22.1, 640 16.5, 16.2, 200 behind 400 16.3, 16.7, 64 behind
// 4032 75, 57; 1300 (352 blocks) 31.2, 28.1, 2048 (512) 51.3, 48, 3000 (768) 90, 103;
// 2 x 1024 (512) 30.2, 32.4; 4 x 768 22.2, 24.3; 8 x 900, 8 heads of 256 (512) 49, 56.
// Of 2142 sizes of 64 to 256 columns with up to 512 blocks 1300 have two, one of them 3%
// slower so, and the rule is 1.0% behind the better one of both on average.
static bool two_teams(const PrefillArgs& a, unsigned blocks, bool wide) {
  const bool whole = a.window <= 0 || a.window >= a.S;
  const long longest =
      whole ? a.S : std::min<long>(a.S, (long)a.window + AP_WAVES * 32 - 1);  // keys
  if (blocks <= 256) return longest >= (!wide ? 608 : a.cap.out > 0.0f ? 384 : 512);
  return blocks <= 512 && longest >= 1280 && whole && a.offset == 0;
}

template <int DK, int DV, bool CAP, int NOPE = 0, bool RAGGED = false>
static void attn_prefill_run(const PrefillArgs& a, hipStream_t stream) {
  const unsigned blocks = (unsigned)a.heads * a.tiles;
  if constexpr (!RAGGED) {
    if (two_teams(a, blocks, ap_keys(DK, DV) == 32)) {
      attn_prefill_kernel<DK, DV, CAP, 2, NOPE>
          <<<dim3(blocks), dim3(2 * AP_BLOCK), 0, stream>>>(a);
      return;
    }
  }
  attn_prefill_kernel<DK, DV, CAP, 1, NOPE, RAGGED>
      <<<dim3(blocks), dim3(AP_BLOCK), 0, stream>>>(a);
}

template <int DK, int DV>
static void attn_prefill_go(const PrefillArgs& a, bool cap, hipStream_t stream) {
  if (cap) attn_prefill_run<DK, DV, true>(a, stream);
  else attn_prefill_run<DK, DV, false>(a, stream);
}

// the arguments that follow from sizes and options
static void prefill_setup(PrefillArgs& a, int B, float scale, float softcap,
                          int window, int offset) {
  constexpr float LOG2E = 1.44269504088896340736f;
  a.flip = scale < 0.0f;
  // a scale of zero: hidden scores still have to vanish
  a.c = fmaxf(fabsf(scale) * LOG2E, 1e-30f);
  a.cap = soft_cap(fabsf(scale), softcap);
  if (softcap > 0.0f) a.c = 1.0f;
  a.window = window;
  a.offset = offset;
  a.heads = B * a.Hq;
  a.tiles = (a.T + AP_WAVES * 32 - 1) / (AP_WAVES * 32);
  a.group = 1;
  if (a.heads % 8 == 0)
    for (int g = 8; g > 1 && a.group == 1; g /= 2)
      if (a.heads / 8 % g == 0) a.group = g;
}

// q: strides in elements; k, v [B, Hkv, cap, D]; out [B, T, Hq, Dv].  16-byte
// loads: all bases and the strides of q are multiples of 8 elements.
extern "C" void launch_attn_prefill(const void* q, const void* k, const void* v,
                                    void* out, int B, int Hq, int Hkv, int T,
                                    int S, long q_b, long q_h, long q_t,
                                    long kScap, long vScap, int Dk, int Dv,
                                    float scale, float softcap, int window,
                                    int causal_offset, hipStream_t stream) {
  PrefillArgs a{(const char*)q, (const char*)k, (const char*)v, (char*)out,
                Hq, Hkv, T, S, q_b, q_h, q_t, kScap, vScap};
  prefill_setup(a, B, scale, softcap, window, causal_offset);
  const bool cap = softcap > 0.0f;
#define AP_GO(K, V) if (Dk == K && Dv == V) attn_prefill_go<K, V>(a, cap, stream);
  AP_SIZES(AP_GO)
#undef AP_GO
}

// Latent attention of a prompt.  Keys and values put together first, queries turned
// and concatenated first, were nine passes over memory; 64 prompts of 512, 16 heads:
// 1.2 ms a layer in all, now 210 us here (175 with whole rows of keys, which lie
// closer) and 26 in mla_rows.
//
// Keys of 128 + 64 columns and values of 128.  q:
// strides in elements; kv [B, S, H, 256]; cache [B, cap, width], whose last 64
// columns are the rotated key part; out [B, T, H, 128].
extern "C" void launch_mla_prompt(const void* q, const void* kv, const void* cache,
                                  const float* cos, const float* sin, void* out,
                                  int B, int H, int T, int S, long q_b, long q_h,
                                  long q_t, long cap, int width, float scale,
                                  int causal_offset, hipStream_t stream) {
  PrefillArgs a{(const char*)q, (const char*)kv, nullptr, (char*)out,
                H, H, T, S, q_b, q_h, q_t};
  a.pe = (const char*)cache + (width - 64) * 2;
  a.pe_b = cap * width * 2;
  a.pe_row = width * 2;
  a.kv_row = H * 256 * 2;
  a.cos = cos;
  a.sin = sin;
  prefill_setup(a, B, scale, 0.0f, 0, causal_offset);
  attn_prefill_run<192, 128, false, 128>(a, stream);
}

// The same for portions of a batch: q rows [dq = 192], turned; k [keys, H * 128], v
// [keys, H * 128], rows [keys, width], whose last 64 columns are the rotated key part;
// out [tokens, H * 128].  2 x 4001 tokens of 16 heads: 275 us, 604 in the general kernel
// (16x16x32 products, tiles through registers, nothing on its way meanwhile).
extern "C" void launch_latent_prompt(const void* q, const void* k, const void* v,
                                     const void* rows, void* out,
                                     const int* portions, const int* cu,
                                     const int* pos0, const int* cuk, int n_short,
                                     int tok_base, int n_tiles, int H, long q_t,
                                     int width, float scale, hipStream_t stream) {
  PrefillArgs a{(const char*)q, (const char*)k, (const char*)v, (char*)out,
                H, H, 1, 1, 0, 192, q_t};
  a.pe = (const char*)rows + (width - 64) * 2;
  a.pe_row = width * 2;
  a.kv_row = a.v_row = H * 128 * 2;
  a.portions = portions;
  a.cu = cu;
  a.pos0 = pos0;
  a.cuk = cuk;
  a.n_short = n_short;
  a.tok_base = tok_base;
  prefill_setup(a, 1, scale, 0.0f, 0, 0);
  a.tiles = n_tiles;
  attn_prefill_run<192, 128, false, 128, true>(a, stream);
}

// ---------------------------------------------------------------------------
// Fragment-layout probe: D = A @ B for one 16x32 @ 32x16 mfma, using the
// maps documented above.  The numerics test compares against torch.matmul
// with asymmetric operands (guide G9: transpose-detecting).
// ---------------------------------------------------------------------------
__global__ void mfma_probe_kernel(const short* __restrict__ A,  // [16][32]
                                  const short* __restrict__ Bm, // [32][16]
                                  float* __restrict__ D) {      // [16][16]
  const int lane = threadIdx.x & (WAVE - 1);
  bf16x8_t a, b;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    a[j] = *reinterpret_cast<const __bf16*>(A + (lane & 15) * 32 + (lane >> 4) * 8 + j);
    b[j] = *reinterpret_cast<const __bf16*>(Bm + ((lane >> 4) * 8 + j) * 16 + (lane & 15));
  }
  f32x4 c = {0, 0, 0, 0};
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
#pragma unroll
  for (int reg = 0; reg < 4; ++reg)
    D[((lane >> 4) * 4 + reg) * 16 + (lane & 15)] = c[reg];
}

extern "C" void launch_mfma_probe(const void* A, const void* Bm, float* D,
                                  hipStream_t stream) {
  mfma_probe_kernel<<<dim3(1), dim3(64), 0, stream>>>(
      (const short*)A, (const short*)Bm, D);
}
