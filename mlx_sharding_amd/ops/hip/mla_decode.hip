// Latent attention of one token per sequence, before and after the attention over
// cached rows [latent | rotated key part] (attn_decode.hip).
//
//   mla_prepare  queries into the space of the cached rows, [W_uk^T q | rotated
//                part], and the token's own row, normed and rotated, into the cache
//   mla_finish   slices of the keys merged, and W_uv of every head's latent
//
// Both are latency: each head's matrix is 128 KB and all of them pass in under a
// microsecond; as separate products, copies, rotations and norms they were twelve
// kernels of 4 to 13 us.  A block takes 16 tokens of one head, a wave 16 rows of
// its matrix, read with the contraction contiguous ([head, row, contraction]).
// Measured: a step of one sequence through four layers of 16 heads, experts and a
// vocabulary of 12800 473 -> 385 us, of 64 sequences 943 -> 784.

#include "mla_decode.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

#define MD_WAVES 4
#define MD_BLOCK (MD_WAVES * WAVE)

__device__ __forceinline__ void turn_pair(float& a, float& b, float c, float s) {
  const float x = a * c - b * s;
  b = b * c + a * s;
  a = x;
}

// grid: (heads x blocks of 64 latent columns, tiles of 16 tokens), then N blocks
// for the cached rows
__global__ __launch_bounds__(MD_BLOCK) void mla_prepare_kernel(
    const MlaPrepareArgs a) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int row_w = a.rank + a.rope;
  const int cols = (a.rank + 63) / 64, tiles = (a.N + 15) / 16;
  const int products = a.heads * cols * tiles;
  if ((int)blockIdx.x >= products) {
    // one token's row: waves share the columns
    __shared__ float scratch[MD_WAVES];
    const int t = blockIdx.x - products;
    const __bf16* c = a.latent + (long)t * a.ld_latent;
    float ss = 0.0f;
    for (int i = threadIdx.x; i < a.rank; i += MD_BLOCK) {
      const float f = (float)c[i];
      ss = fmaf(f, f, ss);
    }
    ss = block_sum<MD_BLOCK>(ss, scratch);
    const float f = rsqrtf(ss / a.rank + a.eps);
    const long pos = a.pos ? *a.pos : a.pos0;
    if (pos >= a.cap) return;
    __bf16* row = a.cache + ((long)t * a.cap + pos) * row_w;
    for (int i = threadIdx.x; i < a.rank; i += MD_BLOCK)
      row[i] = (__bf16)((float)c[i] * f * ((float)a.norm[i] + a.offset));
    for (int i = threadIdx.x; i < a.rope / 2; i += MD_BLOCK) {
      float u = (float)c[a.rank + 2 * i], v = (float)c[a.rank + 2 * i + 1];
      turn_pair(u, v, a.cos[i], a.sin[i]);
      row[a.rank + 2 * i] = (__bf16)u;
      row[a.rank + 2 * i + 1] = (__bf16)v;
    }
    return;
  }
  const int l16 = lane & 15, lg = lane >> 4;
  const int h = blockIdx.x % a.heads;
  const int cb = blockIdx.x / a.heads % cols, tile = blockIdx.x / a.heads / cols;
  const int tok = min(tile * 16 + l16, a.N - 1);
  const long q_head = (long)h * (a.nope + a.rope);
  const int r0 = cb * 64 + wid * 16;
  if (r0 < a.rank) {
    const __bf16* w = a.w + ((long)h * a.rank + min(r0 + l16, a.rank - 1)) * a.nope +
                      lg * 8;
    const __bf16* q = a.q + (long)tok * a.ld_q + q_head + lg * 8;
    f32x4 acc = {0, 0, 0, 0};
    for (int k = 0; k < a.nope; k += 128) {
      bf16x8_t wf[4], qf[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (k + i * 32 < a.nope) {
          wf[i] = *reinterpret_cast<const bf16x8_t*>(w + k + i * 32);
          qf[i] = *reinterpret_cast<const bf16x8_t*>(q + k + i * 32);
        }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (k + i * 32 < a.nope)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i], qf[i], acc, 0, 0, 0);
    }
    if (tile * 16 + l16 < a.N) {
      bf16x4_t o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = (__bf16)acc[j];
      *reinterpret_cast<bf16x4_t*>(a.out + ((long)tok * a.heads + h) * row_w + r0 +
                                   lg * 4) = o;
    }
  }
  if (cb != 0) return;
  // the rotated part of these 16 queries
  for (int i = threadIdx.x; i < 16 * a.rope / 2; i += MD_BLOCK) {
    const int t = tile * 16 + i / (a.rope / 2), p = i % (a.rope / 2);
    if (t >= a.N) break;
    const __bf16* q = a.q + (long)t * a.ld_q + q_head + a.nope + 2 * p;
    float u = (float)q[0], v = (float)q[1];
    turn_pair(u, v, a.cos[p], a.sin[p]);
    __bf16* o = a.out + ((long)t * a.heads + h) * row_w + a.rank + 2 * p;
    o[0] = (__bf16)u;
    o[1] = (__bf16)v;
  }
}

// grid: (heads, tiles of 16 tokens, parts of a head's output columns)
// Bound by the trips to memory that follow one another, and by what a CU reads: the
// slices' maxima, the first partial results and the first rows of the matrix are under
// way together, slices that hold no keys are left out, and where the tokens leave threads
// over, groups of them share a token's slices.  64 slices of 5 tokens 12.5 -> 11.5 us, 32 of
// 16 as fast (13.8), 17 (32 before) 14.3 -> 8.6; with the attention before it one token of
// 3001 keys 14.4 -> 12.7, of 577 11.4 -> 10.8, 128 tokens of 577 34.6 -> 31.4.
__global__ __launch_bounds__(512) void mla_finish_kernel(const MlaFinishArgs a) {
  // a token's latent [16][rank + 8] in bf16: the odd stride keeps the 16 rows that
  // a read meets in different banks
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __bf16* lat = reinterpret_cast<__bf16*>(smem);
  __shared__ float weight[16][64];
  __shared__ f32x4 sums[512];
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int h = blockIdx.x, t0 = blockIdx.y * 16, n = a.slices;
  // Slices behind the keys are empty: the keys there are now may be fewer than those
  // the slices were counted for.  Up to 8 are asked for at once anyway, with no wait for
  // the count (an empty one has weight zero).
  int used = n;
  if (n > 8) {
    const int keys = max(1, a.pos ? min(*a.pos + 1, a.keys) : a.keys);
    const int per = ((keys + n - 1) / n + a.tile - 1) / a.tile * a.tile;
    used = min(n, (keys + per - 1) / per);
  }
  const int stride = a.rank + 8;
  const int part = (a.vdim / 16 + gridDim.z - 1) / gridDim.z * 16;
  const int first = blockIdx.z * part + wid * 16;
  const int last = min(a.vdim, (int)(blockIdx.z + 1) * part);
  const int l16 = lane & 15, lg = lane >> 4;
  auto rows = [&](int r0) {
    return a.w + ((long)h * a.vdim + r0 + l16) * a.rank + lg * 8;
  };
  bf16x8_t wf[16];
  auto fetch = [&](const __bf16* w, int k) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (k + i * 32 < a.rank)
        wf[i] = *reinterpret_cast<const bf16x8_t*>(w + k + i * 32);
  };
  // Asked for together: maxima and sums of the slices, the first partial results and
  // the first rows of the matrix.
  float ml[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const long row = (long)min(t0 + wid + i * 8, a.N - 1) * a.heads + h;
    const float* p = a.part_ml + (row * n + min(lane, used - 1)) * 2;
    ml[i][0] = p[0];
    ml[i][1] = p[1];
  }
  auto weigh = [&] {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float m = lane < used ? ml[i][0] : -1e30f;
      const float l = lane < used ? ml[i][1] : 0.0f;
      const float top = wave_max(m);
      const float e = __builtin_amdgcn_exp2f(m - top);
      weight[wid + i * 8][lane] = e / wave_sum(l * e);
    }
    __syncthreads();
  };
  // Four columns of a token are an item; with few of them groups of threads share the
  // slices, four or more each, and the first adds up.  Loads past the last slice repeat
  // it: left out by branches they cost more (64 tokens: 26.9 us, 22.4 so).
  const int quads = a.rank / 4, items = min(16, a.N - t0) * quads;
  auto over = [](int x, int by) {  // below 2^16
    return (int)(((float)x + 0.5f) * __builtin_amdgcn_rcpf((float)by));
  };
  int groups = 1;
  while (groups * 2 * items <= 512 && groups * 8 <= used) groups *= 2;
  struct Item {
    int t, d;
    const float* p;
  };
  auto item_of = [&](int i) {
    Item x;
    x.t = over(i, quads);
    x.d = (i - x.t * quads) * 4;
    x.p = a.part_o + ((long)(t0 + x.t) * a.heads + h) * n * a.rank + x.d;
    return x;
  };
  auto load = [&](auto& v, const Item& x, int s, int end) {
    constexpr int PER = sizeof(v) / sizeof(v[0]);
#pragma unroll
    for (int j = 0; j < PER; ++j)
      v[j] = *reinterpret_cast<const f32x4*>(x.p + (long)min(s + j, end - 1) * a.rank);
  };
  auto add = [&](f32x4& o, const auto& v, const Item& x, int s, int end) {
    constexpr int PER = sizeof(v) / sizeof(v[0]);
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (s + j < end) {
        const float f = weight[x.t][s + j];
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k] += v[j][k] * f;
      }
  };
  auto keep = [&](const Item& x, f32x4 o) {
    bf16x4_t r;
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = (__bf16)o[j];
    *reinterpret_cast<bf16x4_t*>(lat + x.t * stride + x.d) = r;
  };
  // Of an item the slices from s on, eight more on their way.  Sums of whole eights have
  // no conditions, which their loads would wait for one by one.
  auto eight = [&](f32x4& o, const f32x4 (&v)[8], const Item& x, int s) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float f = weight[x.t][s + j];
#pragma unroll
      for (int k = 0; k < 4; ++k) o[k] += v[j][k] * f;
    }
  };
  auto total = [&](f32x4 (&v)[8], const Item& x, int s, int end) {
    f32x4 u[8], o = {0, 0, 0, 0};
    for (; s + 16 <= end; s += 16) {
      load(u, x, s + 8, end);
      eight(o, v, x, s);
      if (s + 16 < end) load(v, x, s + 16, end);
      eight(o, u, x, s + 8);
    }
    if (s + 8 < end) load(u, x, s + 8, end);
    if (s + 8 <= end) eight(o, v, x, s);
    else add(o, v, x, s, end);
    if (s + 8 < end) add(o, u, x, s + 8, end);
    return o;
  };
  f32x4 v[8];
  if (groups > 1) {
    const int g = over(threadIdx.x, items), share = (used + groups - 1) / groups;
    const Item x = item_of(g < groups ? (int)threadIdx.x - g * items : 0);
    const int end = g < groups ? min(used, (g + 1) * share) : 0, s = g * share;
    load(v, x, min(s, used - 1), max(end, 1));
    if (first < last) fetch(rows(first), 0);
    weigh();
    f32x4 o = total(v, x, s, end);
    sums[threadIdx.x] = o;
    __syncthreads();
    if (g == 0) {
      for (int k = 1; k < groups; ++k) {
        const f32x4 u = sums[k * items + threadIdx.x];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] += u[j];
      }
      keep(x, o);
    }
  } else {
    Item x = item_of(min((int)threadIdx.x, items - 1));
    load(v, x, 0, used);
    if (first < last) fetch(rows(first), 0);
    weigh();
    for (int i = threadIdx.x; i < items;) {
      keep(x, total(v, x, 0, used));
      i += 512;
      if (i < items) {
        x = item_of(i);
        load(v, x, 0, used);
      }
    }
  }
  __syncthreads();
  const int tok = min(l16, a.N - 1 - t0);
  const __bf16* x = lat + tok * stride + lg * 8;
  for (int r0 = first; r0 < last; r0 += 128) {
    f32x4 acc = {0, 0, 0, 0};
    for (int k = 0; k < a.rank; k += 512) {
      if (r0 + k != first) fetch(rows(r0), k);
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (k + i * 32 < a.rank)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              wf[i], *reinterpret_cast<const bf16x8_t*>(x + k + i * 32), acc, 0,
              0, 0);
    }
    if (t0 + l16 >= a.N) continue;
    bf16x4_t o;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = (__bf16)acc[j];
    *reinterpret_cast<bf16x4_t*>(a.out + ((long)(t0 + l16) * a.heads + h) * a.vdim +
                                 r0 + lg * 4) = o;
  }
}

// Rows of a prompt into the cache, normed and rotated, and (rows) once more side by
// side for the projection to keys and values.  A wave per token.
__global__ __launch_bounds__(MD_BLOCK) void mla_rows_kernel(const MlaRowsArgs a) {
  const int lane = threadIdx.x & (WAVE - 1);
  const long n = (long)blockIdx.x * MD_WAVES + threadIdx.x / WAVE;
  if (n >= a.N) return;
  const int t = (int)(n % a.T), width = a.rank + a.rope;
  const __bf16* c = a.latent + n * a.ld_latent;
  __bf16* row = a.cache + (n / a.T * a.cap + a.pos0 + t) * width;
  auto vec = [](const __bf16* p) { return *reinterpret_cast<const bf16x8_t*>(p); };
  float ss = 0.0f;
  for (int i = lane * 8; i < a.rank; i += WAVE * 8) {
    const bf16x8_t x = vec(c + i);
#pragma unroll
    for (int j = 0; j < 8; ++j) ss = fmaf((float)x[j], (float)x[j], ss);
  }
  const float f = rsqrtf(wave_sum(ss) / a.rank + a.eps);
  for (int i = lane * 8; i < a.rank; i += WAVE * 8) {
    const bf16x8_t x = vec(c + i), w = vec(a.norm + i);
    bf16x8_t y;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      y[j] = (__bf16)((float)x[j] * f * ((float)w[j] + a.offset));
    *reinterpret_cast<bf16x8_t*>(row + i) = y;
    if (a.rows) *reinterpret_cast<bf16x8_t*>(a.rows + n * a.rank + i) = y;
  }
  for (int i = lane * 8; i < a.rope; i += WAVE * 8) {
    const bf16x8_t x = vec(c + a.rank + i);
    bf16x8_t y;
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      const long at = ((long)t * a.rope + i + j) / 2;
      float u = (float)x[j], v = (float)x[j + 1];
      turn_pair(u, v, a.cos[at], a.sin[at]);
      y[j] = (__bf16)u;
      y[j + 1] = (__bf16)v;
    }
    *reinterpret_cast<bf16x8_t*>(row + a.rank + i) = y;
  }
}

extern "C" void launch_mla_rows(const MlaRowsArgs* a, hipStream_t stream) {
  mla_rows_kernel<<<dim3((unsigned)((a->N + MD_WAVES - 1) / MD_WAVES)),
                    dim3(MD_BLOCK), 0, stream>>>(*a);
}

extern "C" void launch_mla_prepare(const MlaPrepareArgs* a, hipStream_t stream) {
  const int products = a->heads * ((a->rank + 63) / 64) * ((a->N + 15) / 16);
  mla_prepare_kernel<<<dim3((unsigned)(products + a->N)), dim3(MD_BLOCK), 0,
                       stream>>>(*a);
}

extern "C" void launch_mla_finish(const MlaFinishArgs* a, hipStream_t stream) {
  // A CU reads about 30 bytes a nanosecond: 128 KB of a matrix and 128 KB or more of
  // slices.  Parts share the slices, which then come from L2 (16 heads of 128 x 512, one
  // token and 64; 1, 2, 4, 8 parts: 10.9, 9.0, 8.0, 7.6 us and 10.9, 8.9, 8.3, 12.8).
  const unsigned parts = a->vdim % 64 ? 1 : 4;
  mla_finish_kernel<<<dim3((unsigned)a->heads, (unsigned)((a->N + 15) / 16), parts),
                      dim3(512), (size_t)16 * (a->rank + 8) * 2, stream>>>(*a);
}
