// Flash-decode attention (T=1) over the KV cache — the decode-latency
// hot op (SURVEY.md §7 hard-part #2).
//
// Shapes: q [B, Hq, 1, Dk], kcache [B, Hkv, Scap, Dk], vcache
// [B, Hkv, Scap, Dv]; S = valid length (host int or device pos+1 for
// hipGraph capture).  GQA: one block serves one (batch, kv-head) pair
// and computes all G = Hq/Hkv query heads at once, so each K/V byte is
// read once regardless of the GQA ratio.  Supports MLA shapes (Dk=192,
// Dv=128), gemma2 softcap + sliding window.  fp32 accumulation, online
// softmax over key tiles.
//
// Split-S: at B*Hkv blocks the chip is parallelism-starved (512 blocks
// on 256 CUs), so the key range is split over gridDim.y slices, each
// writing unnormalized partials (m, l, O·l) that a tiny combine kernel
// reduces — flash-decode split-K.  Slice ranges are fractions of the
// CAPACITY so they are static under graph capture; slices past S
// produce (m=-inf, l=0) partials the combiner ignores.
//
// G is a template parameter so per-head register arrays stay statically
// indexed (guide §5.4 rule 20).

#include "hip_common.h"
#include "warm.h"
#include "soft_cap.h"

#include <type_traits>

#define AD_BLOCK 256

// DVT = v-columns per thread (ceil(Dv / AD_BLOCK)): 1 for Dv <= 256,
// 2 for the absorbed-MLA Dv = 512.  vstride is the per-key element
// stride of V rows — for absorbed MLA, V is the first kv_lora_rank
// columns of the K rows themselves (vstride = Dk, vcache = kcache).
template <int G, int DVT>
__global__ __launch_bounds__(AD_BLOCK) void attn_decode_kernel(
    const short* __restrict__ q,      // [B, Hq, Dk]
    const short* __restrict__ kcache, // [B, Hkv, Scap, Dk]
    const short* __restrict__ vcache, // [B, Hkv, Scap, *] (vstride elems/key)
    short* __restrict__ out,          // [B, Hq, Dv]      (nsplit == 1)
    float* __restrict__ part_o,       // [B, Hkv, G, NS, Dv]  (nsplit > 1)
    float* __restrict__ part_ml,      // [B, Hkv, G, NS, 2]
    const int* __restrict__ s_ptr,    // device position (S = *s_ptr + 1), or null
    int B, int Hq, int Hkv, int S, long Scap, int Dk, int Dv, long vstride,
    float scale, float softcap, int window) {
  if (s_ptr) S = *s_ptr + 1;  // hipGraph-captured decode: length lives on device
  const int b = blockIdx.x / Hkv;
  const int hk = blockIdx.x % Hkv;
  const int split = blockIdx.y;
  const int nsplit = gridDim.y;
  // Head-group split (gridDim.z): big-G shapes (absorbed MLA: 16 heads
  // over one KV "head") run as NHG blocks of G heads each — smaller
  // per-block register state → real occupancy; the re-read K tile
  // stays L2-resident.  head id = hk*Gtot + hg*G + g.
  const int hg = blockIdx.z;
  const int Gtot = (Hq / Hkv);
  const int h0 = hk * Gtot + hg * G;
  const int tid = threadIdx.x;

  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  short* q_lds = reinterpret_cast<short*>(smem_raw);           // [G][Dk] bf16
  float* p_lds = reinterpret_cast<float*>(                     // [G][TILE]
      smem_raw + (((size_t)G * Dk * sizeof(short) + 15) & ~(size_t)15));
  float* red = p_lds + (size_t)G * AD_BLOCK;                   // [max(G, NW)]

  for (int i = tid; i < G * Dk; i += AD_BLOCK) {
    int g = i / Dk, d = i % Dk;
    q_lds[i] = q[((long)b * Hq + h0 + g) * Dk + d];
  }
  __syncthreads();

  float m[G], l[G], acc[G * DVT];
#pragma unroll
  for (int g = 0; g < G; ++g) { m[g] = -1e30f; l[g] = 0.0f; }
#pragma unroll
  for (int i = 0; i < G * DVT; ++i) acc[i] = 0.0f;

  const long kbase = ((long)b * Hkv + hk) * Scap;
  int lo = (window > 0 && S > window) ? (S - window) : 0;
  int hi = S;
  if (nsplit > 1) {
    // static tile-aligned slices: capacity-based under graph capture
    // (S lives on device), S-based in eager mode (capacity-based
    // slicing would leave the tail slices empty)
    const long spanc = s_ptr ? Scap : (long)S;
    const long per = ((spanc + nsplit - 1) / nsplit + AD_BLOCK - 1)
                     / AD_BLOCK * AD_BLOCK;
    lo = max((long)lo, per * split);
    hi = min((long)S, per * (split + 1));
  }

  for (int tile = lo; tile < hi; tile += AD_BLOCK) {
    const int s_idx = tile + tid;
    float sc[G];
#pragma unroll
    for (int g = 0; g < G; ++g) sc[g] = -1e30f;
    if (s_idx < hi) {
      const short* krow = kcache + (kbase + s_idx) * Dk;
      float dot[G];
#pragma unroll
      for (int g = 0; g < G; ++g) dot[g] = 0.0f;
      // v_dot2c_f32_bf16: 2 bf16 products + f32 accumulate per VALU op
      // (q stays bf16 in LDS — multiplying bf16 inputs under f32
      // accumulation is numerically identical to the cvt+fma chain).
      // K is loaded in 64-element chunks BEFORE the LDS+dot block:
      // mixing a global load with LDS reads every 8 elements serializes
      // on a per-iteration vmcnt(0) (guide §5 trap 4(b)) — batching the
      // loads keeps 8 of them in flight per wait.
      int d0 = 0;
      for (; d0 + 64 <= Dk; d0 += 64) {
        bf16x8_t kc[8];
#pragma unroll
        for (int c = 0; c < 8; ++c)
          kc[c] = *reinterpret_cast<const bf16x8_t*>(krow + d0 + c * 8);
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
          for (int g = 0; g < G; ++g) {
            bf16x8_t qv = *reinterpret_cast<const bf16x8_t*>(
                q_lds + (size_t)g * Dk + d0 + c * 8);
#pragma unroll
            for (int j = 0; j < 4; ++j)
              dot[g] = dot2_bf16(bf16x2_t{kc[c][2 * j], kc[c][2 * j + 1]},
                                 bf16x2_t{qv[2 * j], qv[2 * j + 1]}, dot[g]);
          }
      }
      for (; d0 < Dk; d0 += 8) {  // Dk % 64 tail (Dk % 8 == 0)
        bf16x8_t kv = *reinterpret_cast<const bf16x8_t*>(krow + d0);
#pragma unroll
        for (int g = 0; g < G; ++g) {
          bf16x8_t qv =
              *reinterpret_cast<const bf16x8_t*>(q_lds + (size_t)g * Dk + d0);
#pragma unroll
          for (int j = 0; j < 4; ++j)
            dot[g] = dot2_bf16(bf16x2_t{kv[2 * j], kv[2 * j + 1]},
                               bf16x2_t{qv[2 * j], qv[2 * j + 1]}, dot[g]);
        }
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float v = dot[g] * scale;
        if (softcap > 0.0f) v = softcap * tanhf(v / softcap);
        sc[g] = v;
      }
    }
    // Online-softmax reductions for ALL G heads in two staged passes
    // (4 barriers/tile): per-head block_max/block_sum loops cost 4*G
    // barriers and serialize the reductions — here wave w reduces
    // heads w, w+NW, ... in parallel from the staged p_lds rows.
    constexpr int NW = AD_BLOCK / WAVE;
    const int lane = tid & (WAVE - 1);
    const int wid = tid / WAVE;
    float alpha[G];
#pragma unroll
    for (int g = 0; g < G; ++g) p_lds[(size_t)g * AD_BLOCK + tid] = sc[g];
    __syncthreads();
    for (int g = wid; g < G; g += NW) {
      float tm = -1e30f;
#pragma unroll
      for (int i = 0; i < NW; ++i)
        tm = fmaxf(tm, p_lds[(size_t)g * AD_BLOCK + lane + i * WAVE]);
      tm = wave_max(tm);
      if (lane == 0) red[g] = tm;
    }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float mnew = fmaxf(m[g], red[g]);
      alpha[g] = __expf(m[g] - mnew);
      float p = (s_idx < hi && sc[g] > -1e29f) ? __expf(sc[g] - mnew) : 0.0f;
      p_lds[(size_t)g * AD_BLOCK + tid] = p;
      m[g] = mnew;
    }
    __syncthreads();
    for (int g = wid; g < G; g += NW) {
      float ts = 0.0f;
#pragma unroll
      for (int i = 0; i < NW; ++i)
        ts += p_lds[(size_t)g * AD_BLOCK + lane + i * WAVE];
      ts = wave_sum(ts);
      if (lane == 0) red[g] = ts;
    }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < G; ++g) l[g] = l[g] * alpha[g] + red[g];
    const int ntile = min(AD_BLOCK, hi - tile);
    const bf16* vbase = ((const bf16*)vcache) + (kbase + tile) * vstride + tid;
    float o[G * DVT];
#pragma unroll
    for (int i = 0; i < G * DVT; ++i) o[i] = 0.0f;
    if (tid < Dv) {
      // per-u column clamp + mask (loop-invariant: no per-element
      // guarded loads — guide §5 trap 4(c))
      long vcol[DVT];
      float vmask[DVT];
#pragma unroll
      for (int u = 0; u < DVT; ++u) {
        const int dv = tid + u * AD_BLOCK;
        vcol[u] = (dv < Dv) ? dv - tid : 0;
        vmask[u] = (dv < Dv) ? 1.0f : 0.0f;
      }
      // batch 8 keys of V loads per wait (trap 4(b), as in the K loop)
      int t = 0;
      for (; t + 8 <= ntile; t += 8) {
        bf16 raw[8][DVT];
#pragma unroll
        for (int tt = 0; tt < 8; ++tt)
#pragma unroll
          for (int u = 0; u < DVT; ++u)
            raw[tt][u] = vbase[(long)(t + tt) * vstride + vcol[u]];
        // all loads are issued before the first use: left to itself the
        // scheduler may pair every load with its wait
        __builtin_amdgcn_sched_barrier(0);
        float vv8[8][DVT];
#pragma unroll
        for (int tt = 0; tt < 8; ++tt)
#pragma unroll
          for (int u = 0; u < DVT; ++u)
            vv8[tt][u] = vmask[u] * bf2f(raw[tt][u]);
#pragma unroll
        for (int tt = 0; tt < 8; ++tt)
#pragma unroll
          for (int g = 0; g < G; ++g) {
            const float p = p_lds[(size_t)g * AD_BLOCK + t + tt];
#pragma unroll
            for (int u = 0; u < DVT; ++u) o[g * DVT + u] += p * vv8[tt][u];
          }
      }
      for (; t < ntile; ++t) {
#pragma unroll
        for (int u = 0; u < DVT; ++u) {
          const float vv = vmask[u] * bf2f(vbase[(long)t * vstride + vcol[u]]);
#pragma unroll
          for (int g = 0; g < G; ++g)
            o[g * DVT + u] += p_lds[(size_t)g * AD_BLOCK + t] * vv;
        }
      }
    }
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int u = 0; u < DVT; ++u)
        acc[g * DVT + u] = acc[g * DVT + u] * alpha[g] + o[g * DVT + u];
    __syncthreads();
  }

  if (nsplit == 1) {
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int u = 0; u < DVT; ++u) {
        const int dv = tid + u * AD_BLOCK;
        if (dv < Dv)
          ((bf16*)out)[((long)b * Hq + h0 + g) * Dv + dv] =
              f2bf(acc[g * DVT + u] / l[g]);
      }
    return;
  }
  // partials: O unnormalized, plus (m, l)
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int u = 0; u < DVT; ++u) {
      const int dv = tid + u * AD_BLOCK;
      if (dv < Dv) {
        const long base = (((long)b * Hq + h0 + g) * nsplit + split) * Dv;
        part_o[base + dv] = acc[g * DVT + u];
      }
    }
  if (tid == 0) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const long base = (((long)b * Hq + h0 + g) * nsplit + split) * 2;
      part_ml[base + 0] = m[g];
      part_ml[base + 1] = l[g];
    }
  }
}

// Combine: one block per (b, hq); Dv threads reduce NS partials.
__global__ void attn_decode_combine_kernel(
    const float* __restrict__ part_o,  // [B*Hq, NS, Dv]
    const float* __restrict__ part_ml, // [B*Hq, NS, 2]
    short* __restrict__ out,           // [B, Hq, Dv]
    int NS, int Dv) {
  const long bh = blockIdx.x;
  const int tid = threadIdx.x;
  float mstar = -1e30f;
  for (int s = 0; s < NS; ++s)
    mstar = fmaxf(mstar, part_ml[(bh * NS + s) * 2]);
  float lsum = 0.0f;
  for (int s = 0; s < NS; ++s) {
    const float ms = part_ml[(bh * NS + s) * 2];
    const float ls = part_ml[(bh * NS + s) * 2 + 1];
    lsum += ls * __expf(ms - mstar);
  }
  for (int d = tid; d < Dv; d += blockDim.x) {
    float o = 0.0f;
    for (int s = 0; s < NS; ++s) {
      const float ms = part_ml[(bh * NS + s) * 2];
      o += part_o[(bh * NS + s) * Dv + d] * __expf(ms - mstar);
    }
    ((bf16*)out)[bh * Dv + d] = f2bf(o / lsum);
  }
}

extern "C" void launch_attn_decode(const void* q, const void* k, const void* v,
                                   void* out, float* part_o, float* part_ml,
                                   int nsplit, const int* s_ptr, int B, int Hq,
                                   int Hkv, int S, long Scap, int Dk, int Dv,
                                   long vstride, float scale, float softcap,
                                   int window, hipStream_t stream) {
  const int Gtot = Hq / Hkv;
  const int DVT = (Dv + AD_BLOCK - 1) / AD_BLOCK;
  // Big-G over few KV heads (absorbed MLA): split heads across
  // gridDim.z — smaller per-block register state, full-chip grids, K
  // tiles re-read from L2 by the sibling head-groups.  8-head groups
  // halve the K re-reads of the round-1 4-head choice at similar
  // occupancy (A/B'd on hardware).
  const int G = (Gtot == 16 && DVT == 2) ? 8 : Gtot;  // 16: -2% (A/B)
  const int NHG = Gtot / G;
  const int nred = (G > AD_BLOCK / WAVE) ? G : AD_BLOCK / WAVE;
  size_t smem = (((size_t)G * Dk * sizeof(short) + 15) & ~(size_t)15) +
                ((size_t)G * AD_BLOCK + nred) * sizeof(float);
  dim3 grid((unsigned)(B * Hkv), (unsigned)nsplit, (unsigned)NHG);
  dim3 block(AD_BLOCK);
#define AD_CASE(GG, VT)                                                      \
  case GG * 16 + VT:                                                         \
    attn_decode_kernel<GG, VT><<<grid, block, smem, stream>>>(               \
        (const short*)q, (const short*)k, (const short*)v, (short*)out,      \
        part_o, part_ml, s_ptr, B, Hq, Hkv, S, Scap, Dk, Dv, vstride, scale, \
        softcap, window);                                                    \
    break;
  switch (G * 16 + DVT) {
    AD_CASE(1, 1)
    AD_CASE(2, 1)
    AD_CASE(4, 1)
    AD_CASE(4, 2)  // absorbed MLA head-group variants, Dv = rank = 512
    AD_CASE(8, 2)
    AD_CASE(16, 2)
    AD_CASE(6, 1)
    AD_CASE(7, 1)  // qwen2 (28 q / 4 kv)
    AD_CASE(8, 1)
    AD_CASE(16, 1)
    default:
      break;
  }
#undef AD_CASE
  if (nsplit > 1) {
    attn_decode_combine_kernel<<<dim3((unsigned)(B * Hq)), dim3(128), 0,
                                 stream>>>(part_o, part_ml, (short*)out,
                                           nsplit, Dv);
  }
}

extern "C" bool attn_decode_supported_shape(int G, int Dv) {
  if (Dv > 512) return false;
  const int dvt = (Dv + AD_BLOCK - 1) / AD_BLOCK;
  if (dvt == 2) return G == 16 || G == 4;
  return G == 1 || G == 2 || G == 4 || G == 6 || G == 7 || G == 8 ||
         G == 16;
}

// ---------------------------------------------------------------------------
// The same on matrix cores, for the head sizes that models have.
//
// A block serves all (up to 16) query heads of one key/value head over a slice
// of its keys.  Tiles of keys and values go to LDS without passing registers, the
// next one while this one is worked on; what it reads from memory is all that
// bounds it, and two blocks a CU keep 64 KB and more in flight.  S^T = K Q^T on
// 16x16x32 products: a wave takes 16 keys (with tiles of 32 keys also half of the
// contraction), leaves its scores in LDS, and after a barrier every wave has the
// weights of the whole tile in the layout of the next product's operand and makes
// a quarter of the output's columns, O^T = V^T P^T.  So waves share no outputs.
// V^T is read by ds_read_b64_tr_b16 out of rows as they lie in memory; values that
// lie in the keys' rows (a cached latent) are staged once for both.
// Weights stay 32-bit: three bf16 parts hold all of their 24 bits, at three times the
// products, which have time to spare (the first size below: 2 us more than with two
// parts, which keep 16 bits, and 3 less than with parts that are rounded, not cut off).
// Slices come from the length on the device, so they are even under capture.
// Measured (before: dot products and sums on the vector units, up to 8 slices of
// the capacity): 64 sequences of 2049 keys, 32 heads of 128 over 8: 179 -> 98 us
// (5.5 TB/s); one of 1024: 24 -> 7.2; 5 of 5004, 16 heads of 256 over 8, capped: 91 ->
// 45; 16 heads over a latent of 576/512, 64 x 513 keys: 66 -> 22, 1 x 3002: 75 -> 13.
// ---------------------------------------------------------------------------

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

#define DT_MAXSPLIT 64

struct DecodeArgs {
  const char *q, *k, *v;   // rows: q [B, Hq, DK], k, v [B, Hkv, cap, *]
  char* out;               // null: one slice is left as a partial result, too
  float *part_o, *part_ml; // [B * Hq, nsplit, DV], [B * Hq, nsplit, 2]
  const int* s_ptr;
  int Hq, Hkv, S, nsplit, window;
  long cap;
  SoftCap score;           // scale and cap
  // a whole step: q and the token's key and value as the projections left them, rows of
  // qs, ks and vs elements from one sequence to the next; rotations; a number per
  // (sequence, key/value head) that is 0 before and after
  const char *knew, *vnew;
  long qs, ks, vs;
  const float *cos, *sin;  // [DK / 2]
  unsigned* tickets;
  Warm warm;               // for blocks from slice nsplit on
};

// Keys and values are read once: as a stream (2) they leave the L2 to what is read again
// (64 x 2049 keys 109 -> 101 us, 5 x 5004 of 256 46.5 -> 45.5).  Not by the tiles of a
// block, which few of them come to and to which they may come out of the L2 (latents 16.4
// -> 16.8 as a stream, 512 keys of heads of 64 5.6 -> 5.8).
template <bool STREAM>
__device__ __forceinline__ void dt_to_lds(const char* src, char* dst) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) void*)src,
      (__attribute__((address_space(3))) void*)dst, 16, 0, STREAM ? 2 : 0);
}

// Place of a 16-byte piece within its row in LDS: keys are read a row a lane,
// values four rows by 32 bytes a quarter wave.
template <int N, bool KEYS>
__device__ __forceinline__ int dt_place(int row, int piece) {
  if (KEYS) return piece ^ (row & 7);
  return N >= 16 ? piece ^ ((row & 7) << 1) : piece ^ ((row & 3) << 1);
}

// largest of the four lanes that share a column
__device__ __forceinline__ float column_max(float x) {
  x = fmaxf(x, __shfl_xor(x, 16, WAVE));
  return fmaxf(x, __shfl_xor(x, 32, WAVE));
}

// Partial results pass from the blocks of a (sequence, key/value head) to the one of them
// that comes last by accesses of the device's scope, as XCDs have L2s of their own.
typedef unsigned long long u64;
typedef u64 u64x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void leave(float* to, f32x4 v) {
  const u64x2 p = __builtin_bit_cast(u64x2, v);
#pragma unroll
  for (int i = 0; i < 2; ++i)
    __hip_atomic_store(reinterpret_cast<u64*>(to) + i, p[i], __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 found(const float* at) {
  return __hip_atomic_load(reinterpret_cast<const u64*>(at), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}

// 8 dimensions from d on of a head, turned: with those half a head away
template <int D>
__device__ __forceinline__ bf16x8_t turned(const char* head, int d, const DecodeArgs& a) {
  constexpr int HALF = D / 2;
  const int c0 = d & (HALF - 1);
  const bf16x8_t u = *reinterpret_cast<const bf16x8_t*>(head + d * 2);
  const bf16x8_t v = *reinterpret_cast<const bf16x8_t*>(head + (d ^ HALF) * 2);
  const float by = d < HALF ? -1.0f : 1.0f;
  bf16x8_t y;
#pragma unroll
  for (int i = 0; i < 8; i += 4) {
    const f32x4 c = *reinterpret_cast<const f32x4*>(a.cos + c0 + i);
    const f32x4 s = *reinterpret_cast<const f32x4*>(a.sin + c0 + i);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      y[i + j] = (__bf16)((float)u[i + j] * c[j] + by * (float)v[i + j] * s[j]);
  }
  return y;
}

// What a block has of its slice, [column of 16][4] a lane of wave `wid` for head l16, to
// the output or to the partial results; the last block of a STEP merges them.  slices:
// those that have keys.
template <int DV, bool STEP, int N>
__device__ __forceinline__ void finish_slice(const DecodeArgs& a, const f32x4 (&o)[N],
                                             float m, float l, long row0, int G, int wid,
                                             int l16, int lg, int slices) {
  const long row = row0 + l16;
  const int col = wid * N * 16 + lg * 4;
  auto write = [&](long r, int c, const f32x4& v, float f) {
    bf16 w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = f2bf(v[i] * f);
    *reinterpret_cast<short4v*>(a.out + (r * DV + c) * 2) = *reinterpret_cast<short4v*>(w);
  };
  if (slices == 1 && a.out) {
    if (l16 >= G) return;
    const float f = 1.0f / l;
#pragma unroll
    for (int d = 0; d < N; ++d) write(row, col + d * 16, o[d], f);
    return;
  }
  const long part = row * a.nsplit + blockIdx.y;
  if constexpr (!STEP) {
    if (l16 >= G) return;
#pragma unroll
    for (int d = 0; d < N; ++d)
      *reinterpret_cast<f32x4*>(a.part_o + part * DV + col + d * 16) = o[d];
    if (wid == 0 && lg == 0) {
      a.part_ml[part * 2] = m;
      a.part_ml[part * 2 + 1] = l;
    }
  } else {
    if (l16 < G) {
#pragma unroll
      for (int d = 0; d < N; ++d) leave(a.part_o + part * DV + col + d * 16, o[d]);
      if (wid == 0 && lg == 0) {
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        __hip_atomic_store(reinterpret_cast<u64*>(a.part_ml) + part,
                           __builtin_bit_cast(u64, f32x2{m, l}), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __shared__ unsigned before;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
      before = __hip_atomic_fetch_add(a.tickets + blockIdx.x, 1u, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (before + 1 != (unsigned)slices) return;
    if (threadIdx.x == 0)
      __hip_atomic_store(a.tickets + blockIdx.x, 0u, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const int items = G * (DV / 4);  // four columns of a head
    // a thread asks for 16 partial results at once, with their weights: those of so many
    // slices and of as many items as that leaves
    auto merge = [&](auto at_once) {
      constexpr int PER = decltype(at_once)::value, AT = 16 / PER;
      for (int i0 = threadIdx.x; i0 < items; i0 += blockDim.x * AT) {
        float top[AT], all[AT];
        f32x4 sum[AT];
#pragma unroll
        for (int t = 0; t < AT; ++t) {
          top[t] = -1e30f;
          all[t] = 0.0f;
          sum[t] = f32x4{0, 0, 0, 0};
        }
        for (int n0 = 0; n0 < slices; n0 += PER) {
          u64x2 v[AT][PER];
          f32x2 ml[AT][PER];
#pragma unroll
          for (int t = 0; t < AT; ++t) {
            const int i = min(i0 + t * (int)blockDim.x, items - 1);
            const long p0 = (row0 + i / (DV / 4)) * a.nsplit;
#pragma unroll
            for (int j = 0; j < PER; ++j) {
              const long n = p0 + min(n0 + j, slices - 1);
              ml[t][j] = __builtin_bit_cast(f32x2, found(a.part_ml + n * 2));
              const float* at = a.part_o + n * DV + i % (DV / 4) * 4;
              v[t][j] = u64x2{found(at), found(at + 2)};
            }
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int t = 0; t < AT; ++t) {
            float most = top[t];
#pragma unroll
            for (int j = 0; j < PER; ++j) most = fmaxf(most, ml[t][j][0]);
            const float keep = __builtin_amdgcn_exp2f(top[t] - most);
            top[t] = most;
            all[t] *= keep;
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[t][r] *= keep;
#pragma unroll
            for (int j = 0; j < PER; ++j) {
              if (n0 + j >= slices) continue;
              const f32x4 f = __builtin_bit_cast(f32x4, v[t][j]);
              const float by = __builtin_amdgcn_exp2f(ml[t][j][0] - most);
              all[t] += ml[t][j][1] * by;
#pragma unroll
              for (int r = 0; r < 4; ++r) sum[t][r] += f[r] * by;
            }
          }
        }
#pragma unroll
        for (int t = 0; t < AT; ++t) {
          const int i = i0 + t * (int)blockDim.x;
          if (i < items)
            write(row0 + i / (DV / 4), i % (DV / 4) * 4, sum[t], 1.0f / all[t]);
        }
      }
    };
    if (slices > 8) merge(std::integral_constant<int, 16>());
    else if (slices > 4) merge(std::integral_constant<int, 8>());
    else merge(std::integral_constant<int, 4>());
  }
}

template <int DK, int DV, int KT, bool INROW>
__global__ __launch_bounds__(AD_BLOCK, 2) void attn_decode_tile_kernel(
    const DecodeArgs a) {
  constexpr int KP = DK / 8, VP = INROW ? KP : DV / 8;  // pieces of a row
  constexpr int NK = DK / 32, ND = DV / 64;
  constexpr int KB = KT * DK * 2, VB = INROW ? 0 : KT * DV * 2;
  constexpr int HALVES = 64 / KT;
  static_assert(KT == 64 || KT == 32, "four waves make the scores of a tile");
  static_assert(NK % HALVES == 0 && KB % 4096 == 0 && VB % 4096 == 0, "sizes");
  __shared__ __attribute__((aligned(16))) char smem[2 * (KB + VB)];
  __shared__ float sc[2][HALVES][KT][16];

  const int S = a.s_ptr ? (int)min((long)*a.s_ptr + 1, a.cap) : a.S;
  const int b = blockIdx.x / a.Hkv, hk = blockIdx.x % a.Hkv;
  const int G = a.Hq / a.Hkv;
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int l16 = lane & 15, lg = lane >> 4;

  const int lo = a.window > 0 && S > a.window ? S - a.window : 0;
  const int per = ((S - lo + a.nsplit - 1) / a.nsplit + KT - 1) / KT * KT;
  const int from = min(S, lo + per * (int)blockIdx.y);
  const int to = min(S, from + per);

  const char* kbase = a.k + (long)blockIdx.x * a.cap * (DK * 2);
  const char* vbase = a.v + (long)blockIdx.x * a.cap * (DV * 2);
  // rows behind the slice repeat its last one; their weights are zero
  auto stage = [&](int t, int buf) {
    char* dst = smem + buf * (KB + VB);
    const char* ks = kbase + (long)t * (DK * 2);
    const char* vs = vbase + (long)t * (DV * 2);
    const int last = to - 1 - t;
#pragma unroll
    for (int i = 0; i < KB / 4096; ++i) {
      const int part = i * 4 + wid, s = part * 64 + lane, row = s / KP;
      dt_to_lds<false>(ks + min(row, last) * (DK * 2) +
                    dt_place<KP, true>(row, s % KP) * 16, dst + part * 1024);
    }
#pragma unroll
    for (int i = 0; i < VB / 4096; ++i) {
      const int part = i * 4 + wid, s = part * 64 + lane, row = s / VP;
      dt_to_lds<false>(vs + min(row, last) * (DV * 2) +
                    dt_place<VP, false>(row, s % VP) * 16,
                dst + KB + part * 1024);
    }
  };
  if (from < to) stage(from, 0);

  const long row0 = (long)b * a.Hq + hk * G;  // first query head
  const int kb = KT == 64 ? wid : wid & 1, half = KT == 64 ? 0 : wid >> 1;
  bf16x8_t qf[NK / HALVES];
  {
    const char* src = a.q + (row0 + min(l16, G - 1)) * (DK * 2) +
                      half * (NK / HALVES) * 64 + lg * 16;
#pragma unroll
    for (int i = 0; i < NK / HALVES; ++i)
      qf[i] = *reinterpret_cast<const bf16x8_t*>(src + i * 64);
  }
  float m = -1e30f, l = 0.0f;  // reference of the exponents (base 2), sum
  f32x4 o[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) o[d] = f32x4{0, 0, 0, 0};

  int buf = 0;
  for (int t = from; t < to; t += KT, buf ^= 1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t + KT < to) stage(t + KT, buf ^ 1);
    const char* kt = smem + buf * (KB + VB);
    const char* vt = kt + KB;
    f32x4 s4 = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < NK / HALVES; ++i) {
      const int piece = (half * (NK / HALVES) + i) * 4 + lg;
      const bf16x8_t f = *reinterpret_cast<const bf16x8_t*>(
          kt + (kb * 16 + l16) * KP * 16 + dt_place<KP, true>(l16, piece) * 16);
      s4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f, qf[i], s4, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) sc[buf][half][kb * 16 + lg * 4 + r][l16] = s4[r];
    __syncthreads();

    float p[KT / 4], top = -INFINITY;  // 8 of every 32 keys
    auto key_of = [&](int i) { return i / 4 * 16 + lg * 4 + (i & 3); };
#pragma unroll
    for (int i = 0; i < KT / 4; ++i) {
      p[i] = sc[buf][0][key_of(i)][l16];
      if (HALVES == 2) p[i] += sc[buf][HALVES - 1][key_of(i)][l16];
    }
    if (a.score.out > 0.0f) {
      soft_capped(a.score, p);
    } else {
#pragma unroll
      for (int i = 0; i < KT / 4; ++i) p[i] *= a.score.lin;
    }
#pragma unroll
    for (int i = 0; i < KT / 4; ++i) {
      if (t + key_of(i) >= to) p[i] = -INFINITY;
      top = fmaxf(top, p[i]);
    }
    top = column_max(top);
    const float m_new = fmaxf(m, top);
    if (__any(m_new > m)) {
      const float f = __builtin_amdgcn_exp2f(m - m_new);
      m = m_new;
      l *= f;
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[d][r] *= f;
    }
#pragma unroll
    for (int x = 0; x < KT / 32; ++x) {
      bf16x8_t v[ND];
      u32x4 w[3];  // pairs: the upper halves of what is left of each weight
#pragma unroll
      for (int j = 0; j < 8; j += 2) {
        float f[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          f[h] = __builtin_amdgcn_exp2f(p[x * 8 + j + h] - m);
          l += f[h];
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const unsigned a = __float_as_uint(f[0]), b = __float_as_uint(f[1]);
          w[i][j / 2] = __builtin_amdgcn_perm(b, a, 0x07060302);
          f[0] -= __uint_as_float(a & 0xFFFF0000u);
          f[1] -= __uint_as_float(b & 0xFFFF0000u);
        }
      }
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        const int row = lg * 4 + (l16 >> 2);  // of this half of 16 keys
        const int piece = (wid * ND + d) * 2 + (l16 >> 1 & 1);
        const char* src = vt + (x * 32 + row) * VP * 16 +
                          dt_place<VP, INROW>(row, piece) * 16 + (l16 & 1) * 8;
        const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(INROW ? src - KB : src));
        const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(
                (INROW ? src - KB : src) + 16 * VP * 16));
        v[d] = __builtin_bit_cast(
            bf16x8_t, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
      }
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int d = 0; d < ND; ++d)
          o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              v[d], __builtin_bit_cast(bf16x8_t, w[i]), o[d], 0, 0, 0);
    }
  }

  l += __shfl_xor(l, 16, WAVE);
  l += __shfl_xor(l, 32, WAVE);
  finish_slice<DV, false>(a, o, m, l, row0, G, wid, l16, lg, a.nsplit);
}

// Whole steps of heads of 64, 128 and 256, and attention alone where there is much of it
// (attn_decode_wave).  A wave has tiles of 32 keys of its own, which go to its own LDS,
// NB of them by turns, and keeps outputs of all columns: scores come out of the first
// product as the second one takes them, so that waves meet at the end of a slice only, and
// each makes its own keys' weights.  In the kernel above a tile's scores pass two barriers
// and all waves make all weights, a chain of 2 us beside loads of 3.  64 sequences of 2049
// keys, 32 heads of 128 over 8: 101 us there, 92 here (5.8 TB/s); one of 1024: 9.6, 9.8; 5 of
// 5004, 16 of 256 over 8: 45.5, 43.5 (a CU has two waves of those; refills of a tile's
// keys ahead of its values gain nothing).
// STEP: queries and the token's key are turned here, its key and value go to the cache
// and into the last tile, and the last block of a head merges the slices.  The chain
// through memory to that block takes 3 us and 1.3 for what a thread asks for at once, the
// merging kernel 4.5; the rotations 2 to 3 instead of 4.6 in a kernel of their own: one
// sequence of 1024 keys, 32 heads of 128 over 8, 14.1 -> 9.6 us for the three.
// Most of such a step is that chain, with the memory idle: beside few pairs and keys, blocks
// of their own fetch the output projection's weights (warm.h).  A step of that sequence, four
// layers with projections, 408 -> 399 us (attention 9 -> 11, projection 8 -> 5.9), of one of
// 300, heads of 64, 132 -> 128.6; 8 of 1000 over 4 heads of 64 144.5 -> 145, so not for those.
// Random layers with 1.5 MB and more of such weights, by pairs: 1 to 6 .980, 8 .981, 12 .986, 16
// .993 of the time without; by keys: up to .5 MB .988, to 8 MB .980 (linear_own_warm).
#define DW_WAVES 2
#define DW_WARM_PAIRS 16
#define DW_WARM_KEYS (8L << 20)  // bytes of keys and values
template <int D, int NB, bool STEP>
__global__ __launch_bounds__(DW_WAVES* WAVE) void attn_decode_wave_kernel(
    const DecodeArgs a) {
  constexpr int KT = 32, P = D / 8, NK = D / 32, ND = D / 16, BYTES = KT * D * 2;
  constexpr int LOADS = 2 * BYTES / 1024;
  // LDS whose size the compiler knows it guards: a read would wait for all loads to LDS
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int S = a.s_ptr ? (int)min((long)*a.s_ptr + 1, a.cap) : a.S;
  const int b = blockIdx.x / a.Hkv, hk = blockIdx.x % a.Hkv;
  const int G = a.Hq / a.Hkv;
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int l16 = lane & 15, lg = lane >> 4;
  constexpr int SPAN = DW_WAVES * KT;
  const int lo = a.window > 0 && S > a.window ? S - a.window : 0;
  if (STEP && (int)blockIdx.y >= a.nsplit) {
    if ((long)gridDim.x * (S - lo) * (D * 4) > DW_WARM_KEYS) return;  // keys have the memory busy
    const unsigned at =
        (unsigned)(unsigned long long)(const __attribute__((address_space(3))) char*)smem;
    warm_rows(a.warm, blockIdx.y * gridDim.x + blockIdx.x, a.nsplit * gridDim.x,
              gridDim.y * gridDim.x, wid, DW_WAVES, at + wid * 1024);
    return;
  }
  const int per = ((S - lo + a.nsplit - 1) / a.nsplit + SPAN - 1) / SPAN * SPAN;
  const int from = min(S, lo + per * (int)blockIdx.y);
  const int to = min(S, from + per);
  if (STEP && from >= to && from > lo) return;  // nothing of the keys, nor of the count

  char* own = smem + wid * NB * 2 * BYTES;
  const char* kbase = a.k + (long)blockIdx.x * a.cap * (D * 2);
  const char* vbase = a.v + (long)blockIdx.x * a.cap * (D * 2);
  // rows behind the slice repeat its last one; their weights are zero
  auto stage = [&](int t, int buf) {
    char* dst = own + buf * (2 * BYTES);
    const char* ks = kbase + (long)t * (D * 2);
    const char* vs = vbase + (long)t * (D * 2);
    const int last = to - 1 - t;
#pragma unroll
    for (int i = 0; i < BYTES / 1024; ++i) {
      const int at = i * WAVE + lane, row = at / P;
      dt_to_lds<true>(ks + min(row, last) * (D * 2) + dt_place<P, true>(row, at % P) * 16,
                dst + i * 1024);
    }
#pragma unroll
    for (int i = 0; i < BYTES / 1024; ++i) {
      const int at = i * WAVE + lane, row = at / P;
      dt_to_lds<true>(vs + min(row, last) * (D * 2) + dt_place<P, false>(row, at % P) * 16,
                dst + BYTES + i * 1024);
    }
  };
  const int first = from + wid * KT, tiles = max(0, (to - first + SPAN - 1) / SPAN);
  auto tile = [&](int i) { return first + i * SPAN; };
#pragma unroll
  for (int i = 0; i < NB; ++i)
    if (i < tiles) stage(tile(i), i);

  const long row0 = (long)b * a.Hq + hk * G;  // first query head
  bf16x8_t qf[NK];
  {
    const char* head = STEP ? a.q + ((long)b * a.qs + (hk * G + min(l16, G - 1)) * D) * 2
                            : a.q + (row0 + min(l16, G - 1)) * (D * 2);
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      if constexpr (STEP) qf[i] = turned<D>(head, i * 32 + lg * 8, a);
      else qf[i] = *reinterpret_cast<const bf16x8_t*>(head + i * 64 + lg * 16);
    }
  }
  // the token itself, at S - 1; it has no place where the cache is full
  const int tail = (to - 1 - from) / KT;  // the slice's last tile
  const bool newest = STEP && from < to && to == S && tail % DW_WAVES == wid &&
                      (!a.s_ptr || *a.s_ptr < a.cap);
  const int piece = lane % P;  // of its rows
  bf16x8_t fresh_k, fresh_v;
  if (newest) {
    const long at = (long)blockIdx.x * a.cap + S - 1;
    fresh_v = *reinterpret_cast<const bf16x8_t*>(
        a.vnew + ((long)b * a.vs + hk * D + piece * 8) * 2);
    fresh_k = turned<D>(a.knew + ((long)b * a.ks + hk * D) * 2, piece * 8, a);
    if (lane < P) {
      *reinterpret_cast<bf16x8_t*>(const_cast<char*>(a.k) + (at * D + piece * 8) * 2) =
          fresh_k;
      *reinterpret_cast<bf16x8_t*>(const_cast<char*>(a.v) + (at * D + piece * 8) * 2) =
          fresh_v;
    }
  }
  float m = -1e30f, l = 0.0f;  // reference of the exponents (base 2), sum
  f32x4 o[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) o[d] = f32x4{0, 0, 0, 0};
  // waited for here: a wait in the loop would be one for all tiles under way
#pragma unroll
  for (int i = 0; i < NK; ++i) asm volatile("" : "+v"(qf[i]));
  if (newest) asm volatile("" : "+v"(fresh_k), "+v"(fresh_v));

  int buf = 0;
  for (int i = 0; i < tiles; ++i, buf = buf + 1 == NB ? 0 : buf + 1) {
    const int t = tile(i);
    // tiles behind this one stay on their way
    if (i + NB - 1 < tiles)
      asm volatile("s_waitcnt vmcnt(%0)" :: "n"((NB - 1) * LOADS) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    char* kt = own + buf * (2 * BYTES);
    char* vt = kt + BYTES;
    if (newest && t + SPAN >= to) {
      // what came from the token's place in the cache is not there yet, in its row and
      // in those behind, which repeat it
      const int row = S - 1 - t;
      if (lane < P)
        *reinterpret_cast<bf16x8_t*>(kt + row * P * 16 +
                                     dt_place<P, true>(row, piece) * 16) = fresh_k;
      for (int r = row + lane / P; r < KT; r += WAVE / P)
        *reinterpret_cast<bf16x8_t*>(vt + r * P * 16 +
                                     dt_place<P, false>(r, piece) * 16) = fresh_v;
    }
    f32x4 s[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
    for (int i = 0; i < NK; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const bf16x8_t f = *reinterpret_cast<const bf16x8_t*>(
            kt + (h * 16 + l16) * P * 16 + dt_place<P, true>(l16, i * 4 + lg) * 16);
        s[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f, qf[i], s[h], 0, 0, 0);
      }
    float p[8], top = -INFINITY;
    auto key_of = [&](int i) { return i / 4 * 16 + lg * 4 + (i & 3); };
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] = s[i / 4][i & 3];
    if (a.score.out > 0.0f) {
      soft_capped(a.score, p);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) p[i] *= a.score.lin;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (t + key_of(i) >= to) p[i] = -INFINITY;
      top = fmaxf(top, p[i]);
    }
    top = column_max(top);
    const float m_new = fmaxf(m, top);
    if (__any(m_new > m)) {
      const float f = __builtin_amdgcn_exp2f(m - m_new);
      m = m_new;
      l *= f;
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[d][r] *= f;
    }
    u32x4 w[3];  // pairs: the upper halves of what is left of each weight
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      float f[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        f[h] = __builtin_amdgcn_exp2f(p[j + h] - m);
        l += f[h];
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const unsigned a = __float_as_uint(f[0]), b = __float_as_uint(f[1]);
        w[i][j / 2] = __builtin_amdgcn_perm(b, a, 0x07060302);
        f[0] -= __uint_as_float(a & 0xFFFF0000u);
        f[1] -= __uint_as_float(b & 0xFFFF0000u);
      }
    }
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      const int row = lg * 4 + (l16 >> 2);  // of each half of 16 keys
      const char* src = vt + row * P * 16 +
                        dt_place<P, false>(row, d * 2 + (l16 >> 1 & 1)) * 16 + (l16 & 1) * 8;
      const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s16x4*)src);
      const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s16x4*)(src + 16 * P * 16));
      const bf16x8_t v = __builtin_bit_cast(
          bf16x8_t, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
      for (int i = 0; i < 3; ++i)
        o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            v, __builtin_bit_cast(bf16x8_t, w[i]), o[d], 0, 0, 0);
    }
    // all of the tile is read
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (i + NB < tiles) stage(tile(i + NB), buf);
  }
  l += __shfl_xor(l, 16, WAVE);
  l += __shfl_xor(l, 32, WAVE);

  // waves' outputs: each finishes half of the columns
  constexpr int N = ND / DW_WAVES;
  static_assert(DW_WAVES == 2 && NB * 4 * BYTES >= DW_WAVES * (N * 4 + 2) * WAVE * 4, "room");
  f32x4* ro = reinterpret_cast<f32x4*>(smem);                    // [waves][N][lanes]
  float* rm = reinterpret_cast<float*>(ro + DW_WAVES * N * WAVE);  // [waves][2][lanes]
  __syncthreads();
#pragma unroll
  for (int d = 0; d < N; ++d) ro[(wid * N + d) * WAVE + lane] = wid ? o[d] : o[N + d];
  rm[(wid * 2) * WAVE + lane] = m;
  rm[(wid * 2 + 1) * WAVE + lane] = l;
  __syncthreads();
  const float om = rm[(wid ^ 1) * 2 * WAVE + lane], ol = rm[((wid ^ 1) * 2 + 1) * WAVE + lane];
  const float most = fmaxf(m, om);
  const float mine = __builtin_amdgcn_exp2f(m - most), its = __builtin_amdgcn_exp2f(om - most);
  f32x4 mo[N];
#pragma unroll
  for (int d = 0; d < N; ++d) {
    const f32x4 v = ro[((wid ^ 1) * N + d) * WAVE + lane];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      mo[d][r] = (wid ? o[N + d][r] : o[d][r]) * mine + v[r] * its;
  }
  finish_slice<D, STEP>(a, mo, most, l * mine + ol * its, row0, G, wid, l16, lg,
                        STEP ? max(1, (S - lo + per - 1) / max(per, 1)) : a.nsplit);
}

// One block per query head: weighs the slices (an empty one has sum zero) and
// adds them up, four columns a thread.
__global__ __launch_bounds__(128) void attn_decode_merge_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml,
    short* __restrict__ out, int n, int Dv) {
  __shared__ float w[DT_MAXSPLIT];
  const long row = blockIdx.x;
  if (threadIdx.x < WAVE) {
    const int s = threadIdx.x;
    const float ms = s < n ? part_ml[(row * n + s) * 2] : -1e30f;
    const float ls = s < n ? part_ml[(row * n + s) * 2 + 1] : 0.0f;
    const float e = __builtin_amdgcn_exp2f(ms - wave_max(ms));
    w[s] = e / wave_sum(ls * e);
  }
  __syncthreads();
  for (int d = threadIdx.x * 4; d < Dv; d += 512) {
    const float* p = part_o + row * n * Dv + d;
    f32x4 o = {0, 0, 0, 0};
#pragma unroll 8
    for (int s = 0; s < n; ++s) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(p + (long)s * Dv);
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] += v[j] * w[s];
    }
    bf16 r[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = f2bf(o[j]);
    *reinterpret_cast<short4v*>(out + row * Dv + d) =
        *reinterpret_cast<short4v*>(r);
  }
}

// head sizes (keys, values), keys of a tile, values within the keys' rows
#define DT_SIZES(DO)                                                         \
  DO(64, 64, 64, false) DO(128, 128, 64, false) DO(192, 128, 32, false)      \
  DO(256, 256, 32, false) DO(576, 512, 32, true)

extern "C" int attn_decode_tile(int G, int Dk, int Dv, bool inrow) {
  if (G > 16) return 0;
#define DT_HAS(K, V, T, R) if (Dk == K && Dv == V && inrow == R) return T;
  DT_SIZES(DT_HAS)
#undef DT_HAS
  return 0;
}

// Whether attention alone has tiles of a wave.  The kernel's two waves a block are longer at
// one tile of keys, and read faster where a CU has many.  Time of a wave's tiles over a
// block's, by tiles of 64 keys of all pairs: heads of 64, below 64 of them 1.05, 128 to
// 255 .99, above 512 .95 and less; of 128, below 32 1.09, 256 to 511 1.00, above 512 .96, above
// 2048 .85; of 256 1.1 and more for most.
extern "C" bool attn_decode_wave(int D, long pairs, long span) {
  const long tiles = pairs * ((span + 63) / 64);
  return D == 64 ? tiles >= 128 : D == 128 && tiles >= 512;
}

// wave: tiles of a wave, also for a call that is not a whole step
template <int DK, int DV, int KT, bool INROW>
static void attn_decode_tile_go(const DecodeArgs& a, int B, bool wave, hipStream_t stream) {
  const dim3 grid((unsigned)(B * a.Hkv), (unsigned)a.nsplit), block(AD_BLOCK);
  if constexpr (DK == DV) {
    // a wave's tiles: 32 KB, of heads of 256 twice that
    constexpr int NB = DK < 256 ? 256 / DK : 2, smem = DW_WAVES * NB * 2 * 32 * DK * 2;
    // blocks that fetch weights: one a CU, which has room for two (of heads of 256 for one)
    const bool warm = a.warm.w && DK < 256 && grid.x <= DW_WARM_PAIRS && grid.x * grid.y <= 256;
    const dim3 more(grid.x, grid.y + (warm ? (255 + grid.x) / grid.x : 0));
    auto go = [&](auto kernel) {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, smem);
      kernel<<<a.tickets ? more : grid, dim3(DW_WAVES * WAVE), smem, stream>>>(a);
    };
    if (a.tickets) return go(&attn_decode_wave_kernel<DK, NB, true>);
    if constexpr (DK < 256) {
      if (wave) go(&attn_decode_wave_kernel<DK, NB, false>);
    } else {
      wave = false;
    }
  }
  if (!wave) attn_decode_tile_kernel<DK, DV, KT, INROW><<<grid, block, 0, stream>>>(a);
  if (a.nsplit > 1 && a.out)
    attn_decode_merge_kernel<<<dim3((unsigned)(B * a.Hq)), dim3(128), 0,
                               stream>>>(a.part_o, a.part_ml, (short*)a.out,
                                         a.nsplit, DV);
}

static void attn_decode_tile_size(const DecodeArgs& a, int B, int Dk, int Dv, bool inrow,
                                  bool wave, hipStream_t stream) {
#define DT_GO(K, V, T, R)                         \
  if (Dk == K && Dv == V && inrow == R)           \
    attn_decode_tile_go<K, V, T, R>(a, B, wave, stream);
  DT_SIZES(DT_GO)
#undef DT_GO
}

// q [B, Hq, Dk]; all bases are multiples of 16 bytes
extern "C" void launch_attn_decode_tile(
    const void* q, const void* k, const void* v, void* out, float* part_o,
    float* part_ml, int nsplit, const int* s_ptr, int B, int Hq, int Hkv, int S,
    long Scap, int Dk, int Dv, bool inrow, bool wave, float scale, float softcap,
    int window, hipStream_t stream) {
  const DecodeArgs a{(const char*)q, (const char*)k, (const char*)v, (char*)out,
                     part_o, part_ml, s_ptr, Hq, Hkv, S, nsplit, window, Scap,
                     soft_cap(scale, softcap)};
  attn_decode_tile_size(a, B, Dk, Dv, inrow, wave, stream);
}

// A step of one token per sequence: rows of q, k and v with strides of qs, ks and vs
// elements; heads of D elements side by side; caches [B, Hkv, Scap, D].  All rows and
// bases are multiples of 16 bytes; tickets [B * Hkv] are 0.  S: without s_ptr the
// length with the token.
extern "C" void launch_attn_step(const void* q, const void* k, const void* v, long qs,
                                 long ks, long vs, const float* cos, const float* sin,
                                 void* kcache, void* vcache, void* out, float* part_o,
                                 float* part_ml, unsigned* tickets, int nsplit,
                                 const int* s_ptr, int B, int Hq, int Hkv, int S,
                                 long Scap, int D, float scale, float softcap, int window,
                                 const Warm* warm, hipStream_t stream) {
  const DecodeArgs a{(const char*)q, (const char*)kcache, (const char*)vcache, (char*)out,
                     part_o, part_ml, s_ptr, Hq, Hkv, S, nsplit, window, Scap,
                     soft_cap(scale, softcap), (const char*)k, (const char*)v, qs, ks, vs,
                     cos, sin, tickets, *warm};
  attn_decode_tile_size(a, B, D, D, false, true, stream);
}
