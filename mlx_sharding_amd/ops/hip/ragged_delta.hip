// Gated delta rule over a ragged batch, state in slots.
//
//   S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q
//
// with q, k, v behind a short causal convolution and silu, q and k unit
// vectors, and one decay g per head, or one per head and key channel (rows of
// S).  The state [D, V] and everything that enters the recurrence are fp32 in
// either element type.
//
//  * short portions (decoding): one kernel does convolution, norms, gates,
//    recurrence, output norm and gate; the state lives in registers.
//  * long portions: chunks of 64 tokens.  With G the running log decay of the
//    chunk, S0 the state before it, and
//        L[i,j] = beta_i exp(G_i - G_j) k_i.k_j   (j < i)
//        A[i,j] =        exp(G_i - G_j) q_i.k_j   (j <= i)
//    the writes are U = (I + L)^-1 diag(beta) (V - diag(exp G) K S0), the
//    outputs O = diag(exp G) Q S0 + A U, and the next state
//    exp(G_last) S0 + K^T diag(exp(G_last - G)) U.  One kernel makes
//    (I + L)^-1 diag(beta) and A of all chunks at once, a second walks the
//    chunks of a (request, head, 16 or 32 value columns).  Products run on the fp32
//    matrix cores, those of the walk (depths of 32, 64 and 128) as eight products of
//    bf16 parts, no further off than fp32's.
//  * decays per channel: exp(G) is a vector then, and L and A sum
//    k_i[d] k_j[d] exp(G_i[d] - G_j[d]) over channels.  Between the tokens of two
//    neighbouring blocks, with the second block's begin as reference, that is a
//    product of two factors, the decay from there to i and the one from j to
//    there; both are running products of decays of at most 1, so nothing
//    overflows and no difference of large logarithms is taken.  Every pair of a
//    chunk lies in two such blocks of 1, 2, 4, 8, 16 or more tokens.
//
// A request at position 0 starts from a zero state whatever its slot holds.
#include <type_traits>
#include "ragged_common.h"

#define DR_CHUNK 64
#define DR_MAXTAPS 8
#define DR_SHORT 16  // most tokens of a short portion

struct DeltaDims {
  int KH, H, D, V, taps;
  int qc, kc, vc, gc, ac, bc;  // column offsets in a projection row; gate (gc)
  long ystride, zstride;       // and decay (ac) in rows z of their own
  bool channels;               // decays per head and key channel
  bool sigmoid;                // the output gate; else silu
};

__device__ __forceinline__ float log_decay(float a, float A_log, float dt) {
  return -expf(A_log) * softplus_f(a + dt);
}

// the factor of one step
template <typename T>
__device__ __forceinline__ float decay_of(float a, float rate, float dt);
template <>
__device__ __forceinline__ float decay_of<float>(float a, float rate, float dt) {
  return expf(-rate * softplus_of<float>(a + dt));
}
template <>
__device__ __forceinline__ float decay_of<__bf16>(float a, float rate, float dt) {
  return __builtin_amdgcn_exp2f(-1.44269504088896340736f * rate *
                                softplus_of<__bf16>(a + dt));
}

__device__ __forceinline__ float out_gate(float x, bool sigmoid) {
  const float s = sigmoid_f(x);
  return sigmoid ? s : x * s;
}

// ---------------------------------------------------------------------------
// Short portions.  Block = (request, q/k head); its r = H / KH value heads
// follow one another, HP at a time.  Threads: VT along V (power of two), DG groups
// along D, RPT state rows per thread.
//
// Bound by latency: the state of a head, 64 KB, passes in half a microsecond a
// block.  So all that a first token needs is asked for at once, what the convolution
// takes before the state (loads come back in order), heads share their barriers, and
// every wave makes the norms of q and k for itself: three barriers a token.
// Measured (before: heads one after the other, nine barriers and loads behind them):
// 12 requests, 16 q/k heads with 2 value heads of 128 x 128 each, 34 -> 17 us; 16
// requests, 16 heads with decays per channel, 19.4 -> 16.8 (10.8 for one token each).
// ---------------------------------------------------------------------------

// EXACT: the threads tile the state without a remainder.  CH: decays per channel.
template <typename T, int RPT, int NT, bool EXACT, bool CH, int HP>
__global__ __launch_bounds__(NT, EXACT && RPT * HP <= 32 ? 4 : 2) void delta_short_kernel(
    const T* __restrict__ y, const T* __restrict__ z,
    const T* __restrict__ conv_w,
    const T* __restrict__ A_log, const T* __restrict__ dt_bias,
    const T* __restrict__ norm_w, float* __restrict__ state,
    T* __restrict__ conv_state, T* __restrict__ out,
    const int* __restrict__ cu, const int* __restrict__ pos0,
    const int* __restrict__ slots, DeltaDims dm, int VT, float q_scale,
    float eps) {
  const int e = blockIdx.x;
  const int kh = blockIdx.y;
  const int t0 = cu[e];
  const int n = min(cu[e + 1] - t0, DR_SHORT);
  const int first_row = n > 0 ? t0 : 0;  // a portion without tokens may lie at the end
  const bool fresh = pos0[e] == 0;
  const long slot = __builtin_amdgcn_readfirstlane(slots[e]);
  const int D = dm.D, V = dm.V;
  const int DG = NT / VT;
  const int tid = threadIdx.x;
  const int lane = tid & (WAVE - 1);
  const int wid = tid / WAVE;
  const int C = 2 * dm.KH * D + dm.H * V;
  const int hist = dm.taps - 1;

  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* qk = reinterpret_cast<float*>(smem);  // [n][2][D]
  float* vb = qk + (long)n * 2 * D;            // [HP][n][V]
  float* red = vb + (long)HP * n * V;          // [HP][2][DG][VT]
  float* scratch = red + HP * 2 * NT;          // [HP][NT / WAVE]
  float* gd = scratch + HP * (NT / WAVE);      // [HP][n][D], decays per channel

  const int v = tid & (VT - 1);
  const int dg = tid / VT;
  const int d0 = dg * RPT;
  const int rep = dm.H / dm.KH;
  // this thread's part of the heads' states
  float S[HP][RPT];
  auto load_state = [&](int p, int h) {
    // uniform row base + one lane offset: no address per row and lane
    const float* sp = state + ((slot * dm.H + h) * (long)D) * V;
    unsigned at = EXACT ? d0 * V + v : min(d0, D - 1) * V + min(v, V - 1);
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      // rows behind the last one repeat it
      const float x = sp[at];
      S[p][i] = fresh ? 0.0f : x;
      if (EXACT) sp += V;
      else at += d0 + i + 1 < D ? V : 0;
    }
  };

  // convolution + silu of a channel for all n tokens: channels 2 D of q and k, then
  // V of each of the heads from h0 on
  struct Conv {
    T w[DR_MAXTAPS], x[DR_MAXTAPS - 1], first;
  };
  // taps sit at the end of w/x, so the index of the newest is fixed
  const int pad = DR_MAXTAPS - dm.taps;
  auto channel = [&](int i, int h0, int& c, int& col) {
    if (i < 2 * D) {
      const int which = i / D, d = i - which * D;
      c = which * dm.KH * D + kh * D + d;
      col = (which ? dm.kc : dm.qc) + kh * D + d;
    } else {
      c = h0 * V + i - 2 * D;
      col = dm.vc + c;
      c += 2 * dm.KH * D;
    }
  };
  auto fetch = [&](Conv& f, int i, int h0) {
    int c, col;
    channel(i, h0, c, col);
    const T* cs = conv_state + (slot * C + c) * hist;
#pragma unroll
    for (int j = 0; j < DR_MAXTAPS; ++j) {
      f.w[j] = j >= pad ? conv_w[(long)c * dm.taps + j - pad] : (T)0.0f;
      if (j < DR_MAXTAPS - 1) f.x[j] = j >= pad ? cs[j - pad] : (T)0.0f;
    }
    f.first = y[(long)first_row * dm.ystride + col];
  };
  auto convolve = [&](const Conv& f, int i, int h0) {
    int c, col;
    channel(i, h0, c, col);
    float x[DR_MAXTAPS];
#pragma unroll
    for (int j = 0; j < DR_MAXTAPS - 1; ++j) x[j] = fresh ? 0.0f : (float)f.x[j];
    float* dst = qk + i;
    int step = 2 * D;
    if (i >= 2 * D) {
      dst = vb + (long)(i - 2 * D) / V * n * V + (i - 2 * D) % V;
      step = V;
    }
#pragma unroll 1
    for (int t = 0; t < n; ++t) {
      x[DR_MAXTAPS - 1] =
          t ? (float)y[(long)(t0 + t) * dm.ystride + col] : (float)f.first;
      float a = 0.0f;
#pragma unroll
      for (int j = 0; j < DR_MAXTAPS; ++j) a += (float)f.w[j] * x[j];
      dst[(long)t * step] = silu_f(a);
#pragma unroll
      for (int j = 0; j < DR_MAXTAPS - 1; ++j) x[j] = x[j + 1];
    }
    // x[j] now holds the input one step older than slot j + 1: the last
    // taps - 1 inputs are x[pad .. MAXTAPS - 2]
    T* cs = conv_state + (slot * C + c) * hist;
#pragma unroll
    for (int j = 0; j < DR_MAXTAPS - 1; ++j)
      if (j >= pad) cs[j - pad] = (T)x[j];
  };

  const int vc = min(v, V - 1);
  const float nw = (float)norm_w[vc];
  for (int hh = 0; hh < rep; hh += HP) {
    const int h0 = kh * rep + hh;
    const int heads = HP == 1 ? 1 : min(HP, rep - hh);
    const int begin = hh ? 2 * D : 0, end = 2 * D + heads * V;
    Conv first;
    if (begin + tid < end) fetch(first, begin + tid, h0);
    // of the first token: decay, write strength, output gate
    T a_in[HP], b_in[HP], g_in[HP], Al[HP], dt[HP];
    auto inputs = [&](int row) {
      const T* yt = y + (long)row * dm.ystride;
      const T* zt = z + (long)row * dm.zstride;
#pragma unroll
      for (int p = 0; p < HP; ++p) {
        const int h = h0 + min(p, heads - 1);
        a_in[p] = CH ? (T)0.0f : zt[dm.ac + h];
        b_in[p] = yt[dm.bc + h];
        g_in[p] = zt[dm.gc + h * V + vc];
      }
    };
    inputs(first_row);
#pragma unroll
    for (int p = 0; p < HP; ++p) {
      const int h = h0 + min(p, heads - 1);
      Al[p] = A_log[h];
      dt[p] = CH ? (T)0.0f : dt_bias[h];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 0; p < HP; ++p) load_state(p, h0 + min(p, heads - 1));
    __builtin_amdgcn_sched_barrier(0);
    if (hh) __syncthreads();  // the previous heads' values have been read
    if (begin + tid < end) convolve(first, begin + tid, h0);
#pragma unroll 1
    for (int i = begin + tid + NT; i < end; i += NT) {
      Conv f;
      fetch(f, i, h0);
      convolve(f, i, h0);
    }
    if constexpr (CH) {
#pragma unroll 1
      for (int i = tid; i < heads * n * D; i += NT) {
        const int p = i / (n * D), t = i / D - p * n, d = i % D, h = h0 + p;
        gd[i] = decay_of<T>((float)z[(t0 + t) * dm.zstride + dm.ac + h * D + d],
                            expf((float)A_log[h]), (float)dt_bias[h * D + d]);
      }
    }
    __syncthreads();
    for (int t = 0; t < n; ++t) {
      if (t) inputs(t0 + t);
      const float* qr = qk + (long)t * 2 * D;
      const float* kr = qr + D;
      float qq = 0.0f, kk = 0.0f, qd = 0.0f;
      for (int d = lane; d < D; d += WAVE) {
        const float a = qr[d], b = kr[d];
        qq += a * a;
        kk += b * b;
        qd += a * b;
      }
      const float fq = q_scale / sqrtf(wave_sum(qq) + 1e-6f);
      const float fk = 1.0f / sqrtf(wave_sum(kk) + 1e-6f);
      const float kq = wave_sum(qd) * fq * fk;
      float sk[HP], sq[HP];
#pragma unroll
      for (int p = 0; p < HP; ++p) sk[p] = sq[p] = 0.0f;
#pragma unroll
      for (int i = 0; i < RPT; ++i) {
        if (EXACT || d0 + i < D) {
          const float a = qr[d0 + i], b = kr[d0 + i];
#pragma unroll
          for (int p = 0; p < HP; ++p) {
            if (CH) S[p][i] *= gd[(min(p, heads - 1) * n + t) * D + d0 + i];
            sk[p] += S[p][i] * b;
            sq[p] += S[p][i] * a;
          }
        }
      }
#pragma unroll
      for (int p = 0; p < HP; ++p) {
        red[p * 2 * NT + dg * VT + v] = sk[p];
        red[p * 2 * NT + NT + dg * VT + v] = sq[p];
      }
      __syncthreads();
      const bool mine = dg == 0 && v < V;
      float g[HP], u[HP], o[HP];
#pragma unroll
      for (int p = 0; p < HP; ++p) {
        float a = 0.0f, b = 0.0f;
        for (int i = 0; i < DG; ++i) {
          a += red[p * 2 * NT + i * VT + v];
          b += red[p * 2 * NT + NT + i * VT + v];
        }
        g[p] = CH ? 1.0f : expf(log_decay((float)a_in[p], (float)Al[p], (float)dt[p]));
        const float beta = sigmoid_f((float)b_in[p]);
        const float vv =
            v < V ? vb[((long)min(p, heads - 1) * n + t) * V + v] : 0.0f;
        u[p] = beta * (vv - g[p] * a * fk);
        o[p] = g[p] * b * fq + kq * u[p];
        const float ss = wave_sum(mine ? o[p] * o[p] : 0.0f);
        if (lane == 0) scratch[p * (NT / WAVE) + wid] = ss;
      }
#pragma unroll
      for (int i = 0; i < RPT; ++i) {
        if (EXACT || d0 + i < D) {
          const float b = kr[d0 + i] * fk;
#pragma unroll
          for (int p = 0; p < HP; ++p) S[p][i] = g[p] * S[p][i] + b * u[p];
        }
      }
      __syncthreads();
      if (mine) {
#pragma unroll
        for (int p = 0; p < HP; ++p) {
          if (p >= heads) break;
          float ss = 0.0f;
#pragma unroll
          for (int w = 0; w < NT / WAVE; ++w) ss += scratch[p * (NT / WAVE) + w];
          const float gate = out_gate((float)g_in[p], dm.sigmoid);
          out[(long)(t0 + t) * ((long)dm.H * V) + (h0 + p) * V + v] =
              (T)(o[p] / sqrtf(ss / (float)V + eps) * nw * gate);
        }
      }
    }
#pragma unroll
    for (int p = 0; p < HP; ++p) {
      if (p >= heads) break;
      // a base of its own: the addresses of the loads are not kept till here
      int head = (int)slot * dm.H + h0 + p;
      asm volatile("" : "+v"(head));
      float* sp = state + (long)__builtin_amdgcn_readfirstlane(head) * D * V;
      if (EXACT || v < V) {
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
          if (EXACT || d0 + i < D) sp[(unsigned)(d0 * V + v)] = S[p][i];
          sp += V;
        }
      }
    }
  }
}

static int pow2_at_least(int v) {
  int p = 16;
  while (p < v) p *= 2;
  return p;
}

// state rows per thread, or 0 if the head is too large for the kernel
extern "C" int delta_short_rows(int D, int V, int nt) {
  const int vt = pow2_at_least(V);
  if (vt > nt) return 0;
  const int need = (D + nt / vt - 1) / (nt / vt);
  for (int r : {4, 16, 32, 64, 128})
    if (need <= r) return r;
  return 0;
}

#define DR_NT 512

template <typename T, bool CH>
static void delta_short_t(const void* y, const void* z, const void* conv_w,
                          const void* A_log, const void* dt_bias,
                          const void* norm_w, float* state, void* conv_state,
                          void* out, const int* cu, const int* pos0,
                          const int* slots, const DeltaDims& dm, int n_req,
                          int max_len, float eps, hipStream_t stream) {
  const int vt = pow2_at_least(dm.V);
  const int rpt = delta_short_rows(dm.D, dm.V, DR_NT);
  const float q_scale = 1.0f / sqrtf((float)dm.D);
  dim3 grid((unsigned)n_req, (unsigned)dm.KH), block(DR_NT);
  auto bytes = [&](int hp) {
    return ((size_t)max_len * (2 * dm.D + hp * ((CH ? dm.D : 0) + dm.V)) +
            hp * (2 * DR_NT + DR_NT / WAVE)) * sizeof(float);
  };
  // two heads at a time where there are two and what they need fits the registers
  // and a quarter of LDS
  const bool exact = dm.V == vt && dm.D == rpt * (DR_NT / vt);
  const bool pairs = dm.H > dm.KH && exact && rpt <= 32 && bytes(2) <= 40960;
  const size_t smem = bytes(pairs ? 2 : 1);
#define DS_ONE(R, X, P)                                                      \
  do {                                                                       \
    if (smem > 65536)                                                        \
      (void)hipFuncSetAttribute(                                             \
          reinterpret_cast<const void*>(                                     \
              &delta_short_kernel<T, R, DR_NT, X, CH, P>),                   \
          hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);            \
    delta_short_kernel<T, R, DR_NT, X, CH, P><<<grid, block, smem, stream>>>(\
        (const T*)y, (const T*)z, (const T*)conv_w, (const T*)A_log,         \
        (const T*)dt_bias, (const T*)norm_w, state, (T*)conv_state, (T*)out, \
        cu, pos0, slots, dm, vt, q_scale, eps);                              \
  } while (0)
#define DS_GO(R, P)                                                          \
  do {                                                                       \
    if (exact)                                                               \
      DS_ONE(R, true, P);                                                    \
    else                                                                     \
      DS_ONE(R, false, P);                                                   \
  } while (0)
#define DS_PAIR(R)                                                           \
  do {                                                                       \
    if (pairs)                                                               \
      DS_ONE(R, true, 2);                                                    \
    else                                                                     \
      DS_GO(R, 1);                                                           \
  } while (0)
  switch (rpt) {
    case 4: DS_PAIR(4); break;
    case 16: DS_PAIR(16); break;
    case 32: DS_PAIR(32); break;
    case 64: DS_GO(64, 1); break;
    case 128: DS_GO(128, 1); break;
    default: break;
  }
#undef DS_PAIR
#undef DS_GO
#undef DS_ONE
}

extern "C" void launch_delta_short(const void* y, const void* z,
                                   const void* conv_w, const void* A_log,
                                   const void* dt_bias, const void* norm_w,
                                   float* state, void* conv_state, void* out,
                                   const int* cu, const int* pos0,
                                   const int* slots, const DeltaDims* dm,
                                   int n_req, int max_len, float eps, bool f32,
                                   hipStream_t stream) {
#define DS_TYPE(T, CH)                                                        \
  delta_short_t<T, CH>(y, z, conv_w, A_log, dt_bias, norm_w, state,           \
                       conv_state, out, cu, pos0, slots, *dm, n_req, max_len, \
                       eps, stream)
  if (dm->channels) {
    if (f32) DS_TYPE(float, true);
    else DS_TYPE(__bf16, true);
  } else {
    if (f32) DS_TYPE(float, false);
    else DS_TYPE(__bf16, false);
  }
#undef DS_TYPE
}

// ---------------------------------------------------------------------------
// Long portions, step 1: convolution, silu, unit norms, gates.
// q, k -> fp32 [n, KH, Dp] (zero padded), v -> T [n, H, Vp], log decay and
// beta -> fp32 [n, H].  One wave per (16 tokens of a chunk, piece): a piece is
// a q or k head, 64 * CW value channels, or the gates.  A lane keeps its CW
// neighbouring channels' inputs of all 16 tokens and their history in
// registers.  NU: channel groups per lane and q/k head, D <= 64 * CW * NU.  TAPS: the
// number of taps, or DR_MAXTAPS for any (taps that are not there are left out one by
// one, as what they would meet need not be finite).
// Bound by memory and by its instructions in like parts.  Blocks that follow one another
// have neighbouring pieces of one row; one norm's root and quotient serve 16 tokens.
// 8002 tokens of 16 q and k heads and 32 value heads of 128: 143 -> 93 us (3.5 TB/s); with
// the taps chosen in the loop a third of the instructions were that.
// ---------------------------------------------------------------------------

// CW neighbouring elements at once (1 or 2)
template <typename T, int CW>
struct __attribute__((aligned(CW * sizeof(T)))) Lanes {
  T v[CW];
};

template <typename T, int CW>
__device__ __forceinline__ void load_lanes(const T* p, float (&o)[CW]) {
  const Lanes<T, CW> t = *reinterpret_cast<const Lanes<T, CW>*>(p);
#pragma unroll
  for (int k = 0; k < CW; ++k) o[k] = (float)t.v[k];
}

template <typename T, int CW>
__device__ __forceinline__ void store_lanes(T* p, const float (&o)[CW]) {
  Lanes<T, CW> t;
#pragma unroll
  for (int k = 0; k < CW; ++k) t.v[k] = (T)o[k];
  *reinterpret_cast<Lanes<T, CW>*>(p) = t;
}

#define DC_BLOCK 256
#define DC_TT 16
#define DC_SUB (DR_CHUNK / DC_TT)

template <typename T, int NU, int CW, int TAPS>
__global__ __launch_bounds__(DC_BLOCK) void delta_conv_kernel(
    const T* __restrict__ y, const T* __restrict__ conv_w,
    const T* __restrict__ A_log, const T* __restrict__ dt_bias,
    const T* __restrict__ conv_state, float* __restrict__ qo,
    float* __restrict__ ko, T* __restrict__ vo, float* __restrict__ lg,
    float* __restrict__ bt, const int* __restrict__ cu,
    const int* __restrict__ pos0, const int* __restrict__ slots,
    const int* __restrict__ tok_entry, const int* __restrict__ chunks,
    int tok_base, DeltaDims dm, int Dp, int Vp, float q_scale, int groups) {
  const int part = blockIdx.x / groups, group = blockIdx.x - part * groups;
  const int chunk = part / DC_SUB, sub = part % DC_SUB;
  const int t0 = chunks[2 * chunk] + sub * DC_TT;
  const int len = min(DC_TT, chunks[2 * chunk + 1] - sub * DC_TT);
  const int lane = threadIdx.x & (WAVE - 1);
  const int piece = __builtin_amdgcn_readfirstlane(
      group * (DC_BLOCK / WAVE) + threadIdx.x / WAVE);
  const int D = dm.D, V = dm.V;
  const int n_qk = 2 * dm.KH;
  const int n_v = (dm.H * Vp + WAVE * CW - 1) / (WAVE * CW);
  if (len <= 0 || piece > n_qk + n_v) return;
  const long i0 = t0 - tok_base;          // row among the long tokens
  const int e = tok_entry[t0];
  const int rel = t0 - cu[e];             // place within the portion
  const bool fresh = pos0[e] == 0;
  const int taps = TAPS < DR_MAXTAPS ? TAPS : dm.taps, hist = taps - 1;
  const int C = 2 * dm.KH * D + dm.H * V;
  const T* cs = conv_state + (long)slots[e] * C * hist;
  const T* yt = y + (long)t0 * dm.ystride;

  // channels c.. (columns col.. of y): convolved, silu'd values of 16 tokens
  auto convolve = [&](int c, int col, float (&o)[DC_TT][CW]) {
    float x[DC_TT + TAPS - 1][CW], w[TAPS][CW];
#pragma unroll
    for (int k = 0; k < DC_TT + TAPS - 1; ++k) {
      const int t = k - (TAPS - 1);
#pragma unroll
      for (int q = 0; q < CW; ++q) x[k][q] = 0.0f;
      if (t >= 0) {
        // tokens past the end repeat the last one and are not stored
        load_lanes<T, CW>(yt + (long)min(t, len - 1) * dm.ystride + col, x[k]);
      } else if (t >= -hist) {
        if (rel + t >= 0)
          load_lanes<T, CW>(yt + (long)t * dm.ystride + col, x[k]);
        else if (!fresh)
#pragma unroll
          for (int q = 0; q < CW; ++q)
            x[k][q] = (float)cs[(long)(c + q) * hist + hist + rel + t];
      }
    }
    const int pad = TAPS - taps;
#pragma unroll
    for (int j = 0; j < TAPS; ++j)
#pragma unroll
      for (int q = 0; q < CW; ++q)
        w[j][q] = j >= pad ? (float)conv_w[(long)(c + q) * taps + j - pad]
                           : 0.0f;
#pragma unroll
    for (int t = 0; t < DC_TT; ++t)
#pragma unroll
      for (int q = 0; q < CW; ++q) {
        float a = 0.0f;
#pragma unroll
        for (int j = 0; j < TAPS; ++j)
          if (j >= pad) a += w[j][q] * x[t + j][q];
        o[t][q] = silu_f(a);
      }
  };

  if (piece < n_qk) {
    const int which = piece / dm.KH, kh = piece - which * dm.KH;
    float o[NU][DC_TT][CW];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int d = (lane + u * WAVE) * CW;
      if (d < D) {
        convolve(which * dm.KH * D + kh * D + d,
                 (which ? dm.kc : dm.qc) + kh * D + d, o[u]);
      } else {
#pragma unroll
        for (int t = 0; t < DC_TT; ++t)
#pragma unroll
          for (int q = 0; q < CW; ++q) o[u][t][q] = 0.0f;
      }
    }
    float* dst = (which ? ko : qo) + (i0 * dm.KH + kh) * Dp;
    float sq = 0.0f;  // lane t: of token t
#pragma unroll
    for (int t = 0; t < DC_TT; ++t) {
      float ss = 0.0f;
#pragma unroll
      for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int q = 0; q < CW; ++q) ss += o[u][t][q] * o[u][t][q];
      ss = wave_sum(ss);
      if (lane == t) sq = ss;
    }
    const float by = (which ? 1.0f : q_scale) / sqrtf(sq + 1e-6f);
#pragma unroll
    for (int t = 0; t < DC_TT; ++t) {
      const float s = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(by), t));
      if (t < len) {
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          const int d = (lane + u * WAVE) * CW;
#pragma unroll
          for (int q = 0; q < CW; ++q) o[u][t][q] *= s;
          if (d < Dp)
            store_lanes<float, CW>(dst + (long)t * dm.KH * Dp + d, o[u][t]);
        }
      }
    }
  } else if (piece < n_qk + n_v) {
    const int j = ((piece - n_qk) * WAVE + lane) * CW;
    if (j >= dm.H * Vp) return;
    const int h = j / Vp, v = j - h * Vp;
    float o[DC_TT][CW];
    if (v < V) {
      convolve(2 * dm.KH * D + h * V + v, dm.vc + h * V + v, o);
    } else {
#pragma unroll
      for (int t = 0; t < DC_TT; ++t)
#pragma unroll
        for (int q = 0; q < CW; ++q) o[t][q] = 0.0f;
    }
#pragma unroll
    for (int t = 0; t < DC_TT; ++t)
      if (t < len)
        store_lanes<T, CW>(vo + (i0 + t) * ((long)dm.H * Vp) + j, o[t]);
  } else {
    for (int j = lane; j < len * dm.H; j += WAVE) {
      const int t = j / dm.H, h = j - t * dm.H;
      const T* yr = yt + (long)t * dm.ystride;
      if (!dm.channels)
        lg[(i0 + t) * dm.H + h] =
            log_decay((float)yr[dm.ac + h], (float)A_log[h], (float)dt_bias[h]);
      bt[(i0 + t) * dm.H + h] = sigmoid_f((float)yr[dm.bc + h]);
    }
  }
}

// The last taps - 1 inputs of every channel; runs after the convolution.
template <typename T>
__global__ __launch_bounds__(DC_BLOCK) void delta_conv_state_kernel(
    const T* __restrict__ y, T* __restrict__ conv_state,
    const int* __restrict__ cu, const int* __restrict__ pos0,
    const int* __restrict__ slots, int n_short, DeltaDims dm) {
  const int e = n_short + blockIdx.x;
  const int c = blockIdx.y * DC_BLOCK + threadIdx.x;
  const int D = dm.D, V = dm.V;
  const int nq = dm.KH * D;
  const int C = 2 * nq + dm.H * V;
  if (c >= C) return;
  const int col = c < nq ? dm.qc + c
                         : (c < 2 * nq ? dm.kc + c - nq : dm.vc + c - 2 * nq);
  const int hist = dm.taps - 1;
  const int t0 = cu[e], n = cu[e + 1] - t0;
  const bool fresh = pos0[e] == 0;
  T* cs = conv_state + ((long)slots[e] * C + c) * hist;
  for (int j = 0; j < hist; ++j) {  // ascending: reads stay ahead of writes
    const int s = n - hist + j;
    if (s >= 0)
      cs[j] = y[(long)(t0 + s) * dm.ystride + col];
    else
      cs[j] = fresh ? (T)0.0f : cs[hist + s];
  }
}

// ---------------------------------------------------------------------------
// Step 2, all chunks at once.  Block = (chunk, head), 4 waves; wave w makes
// rows 16w..16w+15 of the two Gram matrices and column tile w of the inverse.
//   tm [chunks, H, 64, 64]  (I + L)^-1 diag(beta) (lower tiles only)
//   am [chunks, H, 64, 64]  A (lower tiles only)
//   ge [chunks, H, 2, 64]   exp(G), exp(G_last - G)
// Bound by latency, and by what is written.  Operands are on their way a step ahead, and
// the value heads of a q/k head run on one XCD: 126 chunks of 32 heads 138 -> 110 us; with
// two of them in a block 118 -> 84 (another card, on which that kernel took 118).
// ---------------------------------------------------------------------------

#define DR_LS 68

// Lower tiles of (I + L)^-1 diag(by), by four waves; ls: L, rows of DR_LS, whose
// tiles on the diagonal are overwritten.  A wave inverts one of these by forward
// substitution, a column per lane, and then makes the tiles below it from products,
// X_ij = -X_ii sum_k L_ik X_kj: a product's result lies as the next one's operand.
// One wave for all 64 rows left three idle through a chain four times as long: the
// matrices of 126 chunks, 32 heads 167 -> 138 us, with decays per channel (a mixed
// batch of 16 heads) 58 -> 46.
__device__ __forceinline__ void invert_tiles(float* ls, const float* by, float* tm,
                                             int wid, int lane) {
  const int lr = lane & 15, g4 = lane >> 4;
  float* own = ls + wid * 16 * DR_LS + wid * 16;
  float x[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    float a0 = i == lr ? 1.0f : 0.0f, a1 = 0.0f;
    const float* row = own + i * DR_LS;
#pragma unroll
    for (int j = 0; j + 2 <= i; j += 2) {
      a0 -= row[j] * x[j];
      a1 -= row[j + 1] * x[j + 1];
    }
    if (i & 1) a0 -= row[i - 1] * x[i - 1];
    x[i] = a0 + a1;
  }
  f32x4 d;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    d[r] = g4 < 2 ? (g4 ? x[4 + r] : x[r]) : (g4 == 2 ? x[8 + r] : x[12 + r]);
  const float b = by[wid * 16 + lr];
  auto put = [&](int i, const f32x4& v) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      tm[(i * 16 + g4 * 4 + r) * 64 + wid * 16 + lr] = v[r] * b;
  };
#pragma unroll
  for (int r = 0; r < 4; ++r) own[(g4 * 4 + r) * DR_LS + lr] = d[r];
  put(wid, d);
  __syncthreads();
  f32x4 col[4] = {d, d, d, d};  // tiles of this column, from the diagonal on
#pragma unroll
  for (int i = 1; i < 4; ++i) {
    if (i <= wid) continue;
    const float* row = ls + (i * 16 + lr) * DR_LS + g4 * 4;
    f32x4 sum = {0, 0, 0, 0}, y = {0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < i; ++k) {
      if (k < wid) continue;
      const f32x4 l = load4(row + k * 16);
#pragma unroll
      for (int t = 0; t < 4; ++t) sum = mma4(l[t], col[k][t], sum);
    }
    const f32x4 u = load4(row + i * 16);
#pragma unroll
    for (int t = 0; t < 4; ++t) y = mma4(u[t], -sum[t], y);
    col[i] = y;
    put(i, y);
  }
}

// Value heads of a q/k head that a block makes one after the other, from the same
// products, which are half of a head's work (fp32 matrix cores).  Blocks of one head,
// of two, us: 32 heads over 16, 126 chunks 118, 84, 63 59.8, 47.6, 32 38.1, 25.4, 16 19.2,
// 18.4, 10 (320 blocks) 18.2, 17.3, 5 14.1, 18.1: those leave CUs idle.
#define DC_HEADS 2

__global__ __launch_bounds__(256) void delta_chunk_kernel(
    const float* __restrict__ qn, const float* __restrict__ kn,
    const float* __restrict__ lg, const float* __restrict__ bt,
    float* __restrict__ tm, float* __restrict__ am, float* __restrict__ ge,
    const int* __restrict__ chunks, int n_chunks, int tok_base, int KH, int H, int Dp,
    int per) {
  // blocks go round the XCDs: eight pairs of a chunk and a q/k head, then their next
  // `per` value heads, which read the same rows from the L2 they came to
  const int r = H / KH, g = r / per, round = blockIdx.x / (8 * g);
  const int at = blockIdx.x - round * 8 * g, pair = round * 8 + at % 8;
  if (pair >= n_chunks * KH) return;
  const int c = pair / KH, kh = pair - c * KH, h0 = kh * r + at / 8 * per;
  const int i0 = chunks[2 * c] - tok_base;
  const int len = chunks[2 * c + 1];
  const int tid = threadIdx.x;
  const int lane = tid & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int lr = lane & 15, g4 = lane >> 4;

  __shared__ double gs[DC_HEADS][DR_CHUNK];
  __shared__ float bs[DC_HEADS][DR_CHUNK];
  __shared__ __attribute__((aligned(16))) float ls[DR_CHUNK * DR_LS];

  if (wid < per) {
    const int h = h0 + wid;
    const long ch = (long)c * H + h;
    // running sum of log decays; differences of it must stay exact to fp32,
    // also behind strong decays, hence double
    const bool in = lane < len;
    double g = in ? (double)lg[(long)(i0 + lane) * H + h] : 0.0;
#pragma unroll
    for (int off = 1; off < WAVE; off <<= 1) {
      const double o = __shfl_up(g, off, WAVE);
      if (lane >= off) g += o;
    }
    const double last = __shfl(g, WAVE - 1, WAVE);
    gs[wid][lane] = g;
    bs[wid][lane] = in ? bt[(long)(i0 + lane) * H + h] : 0.0f;
    ge[ch * 128 + lane] = expf((float)g);
    ge[ch * 128 + 64 + lane] = expf((float)(last - g));
  }

  f32x4 kk[4], qk[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    kk[j] = f32x4{0, 0, 0, 0};
    qk[j] = f32x4{0, 0, 0, 0};
  }
  // rows past the end repeat the last one: their beta is 0
  const int ra = min(wid * 16 + lr, len - 1);
  const float* kbase = kn + ((long)i0 * KH + kh) * Dp + g4 * 4;
  const float* qbase = qn + ((long)i0 * KH + kh) * Dp + g4 * 4;
  const long rstride = (long)KH * Dp;
  // one step's operands are on their way while another's are in the matrix cores
  struct Step {
    f32x4 q, k[4];
  };
  auto fetch = [&](Step& f, int d) {
    f.q = load4(qbase + ra * rstride + d);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j <= wid) f.k[j] = load4(kbase + min(j * 16 + lr, len - 1) * rstride + d);
  };
  auto use = [&](const Step& f) {
    const f32x4 ka = wid == 0 ? f.k[0] : wid == 1 ? f.k[1] : wid == 2 ? f.k[2] : f.k[3];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j > wid) continue;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        kk[j] = mma4(ka[s], f.k[j][s], kk[j]);
        qk[j] = mma4(f.q[s], f.k[j][s], qk[j]);
      }
    }
  };
  Step one, two;
  fetch(one, 0);
  for (int d = 0; d < Dp; d += 32) {
    if (d + 16 < Dp) fetch(two, d + 16);
    use(one);
    if (d + 32 < Dp) fetch(one, d + 32);
    if (d + 16 < Dp) use(two);
  }
  __syncthreads();
  for (int n = 0; n < per; ++n) {
    const long ch = (long)c * H + h0 + n;
    if (n) __syncthreads();  // the last head's matrix is read
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j > wid) continue;
      const int col = j * 16 + lr;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = wid * 16 + g4 * 4 + r;
        const float dec = col <= row ? expf((float)(gs[n][row] - gs[n][col])) : 0.0f;
        ls[row * DR_LS + col] = col < row ? bs[n][row] * dec * kk[j][r] : 0.0f;
        am[ch * 4096 + row * 64 + col] = dec * qk[j][r];
      }
    }
    __syncthreads();
    invert_tiles(ls, bs[n], tm + ch * 4096, wid, lane);
  }
}

// The same for decays per channel, and what the walk multiplies the state with:
//   qg, kg [tokens, H, Dp]  q and k with the decay from the chunk's begin
//   kl     [tokens, H, Dp]  k with the decay to the chunk's end
//   gl     [chunks, H, Dp]  the decay of the whole chunk
// Wave w has token rows 16w..16w+15, a lane one of them and four of each 16
// channels.  Per 16 channels, running products over blocks of 1, 2, 4, 8 and 16
// rows grow by one exchange between lanes each: `from` decays from the row's
// block's begin to the row, `to` from the row to its block's end.
#define DCH_STEPS 4                    // steps of 16 channels between barriers
#define DCH_LS (DCH_STEPS * 16 + 4)

// VEC: channels and rows of z are whole vectors of 4.
template <typename T, bool VEC>
__global__ __launch_bounds__(256, 2) void delta_chunk_channels_kernel(
    const float* __restrict__ qn, const float* __restrict__ kn,
    const T* __restrict__ z, const T* __restrict__ A_log,
    const T* __restrict__ dt_bias, const float* __restrict__ bt,
    float* __restrict__ tm, float* __restrict__ am, float* __restrict__ qg,
    float* __restrict__ kg, float* __restrict__ kl, float* __restrict__ gl,
    const int* __restrict__ chunks, int tok_base, DeltaDims dm, int Dp) {
  const int c = blockIdx.x, h = blockIdx.y;
  const int H = dm.H, KH = dm.KH, D = dm.D;
  const int kh = h / (H / KH);
  const int i0 = chunks[2 * c] - tok_base;
  const int len = chunks[2 * c + 1];
  const int tid = threadIdx.x;
  const int lane = tid & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int lr = lane & 15, g4 = lane >> 4;

  __shared__ float bs[DR_CHUNK];
  __shared__ __attribute__((aligned(16))) float ms[4][DCH_STEPS * 16];
  // k with the decay to its wave's last row; later I + L
  __shared__ __attribute__((aligned(16))) float ls[DR_CHUNK * DR_LS];
  static_assert(DCH_LS <= DR_LS, "");

  const long ch = (long)c * H + h;
  if (wid == 0) bs[lane] = lane < len ? bt[(long)(i0 + lane) * H + h] : 0.0f;

  const int row = wid * 16 + lr;
  const bool in = row < len;
  // rows past the end repeat the last one with k = q = 0, decay 1 and beta 0
  const long tok = i0 + min(row, len - 1);
  const float* kp = kn + (tok * KH + kh) * Dp + g4 * 4;
  const float* qp = qn + (tok * KH + kh) * Dp + g4 * 4;
  const T* zp = z + (tok_base + tok) * dm.zstride + dm.ac + (long)h * D;
  const T* dp = dt_bias + (long)h * D;
  const long at = ((long)(i0 + row) * H + h) * Dp + g4 * 4;
  const float rate = expf((float)A_log[h]);
  const f32x4 zero = {0, 0, 0, 0}, one = {1, 1, 1, 1};

  f32x4 kk[4], qk[4], kko[3], qko[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) kk[i] = qk[i] = zero;
#pragma unroll
  for (int i = 0; i < 3; ++i) kko[i] = qko[i] = zero;
  float diag = 0.0f;

  for (int d0 = 0; d0 < Dp; d0 += DCH_STEPS * 16) {
    f32x4 ka[DCH_STEPS], qa[DCH_STEPS], kb[DCH_STEPS];
    f32x4 za[DCH_STEPS], dt[DCH_STEPS];
    // everything a slice reads is asked for first
#pragma unroll
    for (int s = 0; s < DCH_STEPS; ++s) {
      const int ds = min(d0 + s * 16, Dp - 16), d = ds + g4 * 4;
      ka[s] = load4(kp + ds);
      qa[s] = load4(qp + ds);
      if constexpr (VEC) {
        const int dc = min(d, D - 4);
        za[s] = load4(zp + dc);
        dt[s] = load4(dp + dc);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int dc = min(d + j, D - 1);
          za[s][j] = (float)zp[dc];
          dt[s][j] = (float)dp[dc];
        }
      }
    }
#pragma unroll
    for (int s = 0; s < DCH_STEPS; ++s) {
      const int ds = d0 + s * 16;
      if (ds >= Dp) continue;
      const f32x4 k = in ? ka[s] : zero, q = in ? qa[s] : zero;
      f32x4 from, to = one;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float g = decay_of<T>(za[s][j], rate, dt[s][j]);
        from[j] = in && ds + g4 * 4 + j < D ? g : 1.0f;
        diag += q[j] * k[j];
      }
#pragma unroll
      for (int l = 0; l < 4; ++l) {
        const int half = 1 << l;
        const f32x4 kf = k * from, qf = q * from, kt = k * to;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          kk[l] = mma4(kf[j], kt[j], kk[l]);
          qk[l] = mma4(qf[j], kt[j], qk[l]);
        }
        // the other half's whole decay: of the first for rows of the second
        const bool second = lr & half;
        const int src = (lane & ~(2 * half - 1)) + (second ? half : 2 * half) - 1;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float other = __shfl(from[j], src, WAVE);
          if (second) from[j] *= other;
          else to[j] *= other;
        }
      }
      ka[s] = k * from;
      qa[s] = q * from;
      kb[s] = k * to;
      store4(ls + row * DCH_LS + s * 16 + g4 * 4, kb[s]);
      if (lr == 15) store4(&ms[wid][s * 16 + g4 * 4], from);
    }
    __syncthreads();
    // blocks before this wave's, the nearest first
#pragma unroll
    for (int b = 2; b >= 0; --b) {
      if (b >= wid) continue;
#pragma unroll
      for (int s = 0; s < DCH_STEPS; ++s) {
        if (d0 + s * 16 >= Dp) continue;
        const f32x4 k = load4(ls + (b * 16 + lr) * DCH_LS + s * 16 + g4 * 4);
        const f32x4 m = load4(&ms[b][s * 16 + g4 * 4]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          kko[b] = mma4(ka[s][j], k[j], kko[b]);
          qko[b] = mma4(qa[s][j], k[j], qko[b]);
        }
        ka[s] = ka[s] * m;
        qa[s] = qa[s] * m;
      }
    }
    // and those behind it
#pragma unroll
    for (int b = 1; b < 4; ++b) {
      if (b <= wid) continue;
#pragma unroll
      for (int s = 0; s < DCH_STEPS; ++s)
        if (d0 + s * 16 < Dp)
          kb[s] = kb[s] * load4(&ms[b][s * 16 + g4 * 4]);
    }
    if (in) {
#pragma unroll
      for (int s = 0; s < DCH_STEPS; ++s) {
        const int ds = d0 + s * 16;
        if (ds >= Dp) continue;
        store4(kg + at + ds, ka[s]);
        store4(qg + at + ds, qa[s]);
        store4(kl + at + ds, kb[s]);
      }
    }
    if (tid < DCH_STEPS * 16 && d0 + tid < Dp)
      gl[ch * Dp + d0 + tid] =
          (ms[0][tid] * ms[1][tid]) * (ms[2][tid] * ms[3][tid]);
    __syncthreads();
  }
  diag += __shfl_xor(diag, 16, WAVE);
  diag += __shfl_xor(diag, 32, WAVE);  // of this lane's row: q.k

#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = wid * 16 + g4 * 4 + r;
    const float b = bs[i];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      if (j >= wid) continue;
      ls[i * DR_LS + j * 16 + lr] = b * kko[j][r];
      am[ch * 4096 + i * 64 + j * 16 + lr] = qko[j][r];
    }
    // the level that separates the row from the column
    const int local = g4 * 4 + r;
    float kv = 0.0f, qv = local == lr ? diag : 0.0f;
#pragma unroll
    for (int l = 0; l < 4; ++l)
      if (local > lr && (local ^ lr) >> l == 1) {
        kv = kk[l][r];
        qv = qk[l][r];
      }
    ls[i * DR_LS + row] = b * kv;
    am[ch * 4096 + i * 64 + row] = qv;
  }
  __syncthreads();
  invert_tiles(ls, bs, tm + ch * 4096, wid, lane);
}

// ---------------------------------------------------------------------------
// Step 3: the walk.  Block = (value column tile, head, request), 4 waves;
// wave w owns token rows 16w..16w+15 of a chunk and state row tiles w, w+4,...
// A operands come straight from global memory as vectors (the contraction
// order inside 16 is permuted the same way on both sides).  CH: decays per
// channel; q, k and kt (k as the state takes it up) come with their decays, one
// row per value head (KH == H), and ge is the chunk's decay [chunks, H, Dp].
// ---------------------------------------------------------------------------

template <typename T, bool CH>
__global__ __launch_bounds__(256) void delta_walk_kernel(
    const float* __restrict__ qn, const float* __restrict__ kn,
    const float* __restrict__ kt, const T* __restrict__ vn, const float* __restrict__ tm,
    const float* __restrict__ am, const float* __restrict__ ge,
    float* __restrict__ state, float* __restrict__ o,
    const int* __restrict__ chunks, const int* __restrict__ chunk_cu,
    const int* __restrict__ pos0, const int* __restrict__ slots, int n_short,
    int tok_base, int KH, int H, int D, int Dp, int V, int Vp) {
  const int v0 = blockIdx.x * 16;
  const int h = blockIdx.y;
  const int e = blockIdx.z;
  const int kh = h / (H / KH);
  const int tid = threadIdx.x;
  const int lane = tid & (WAVE - 1);
  const int wid = tid / WAVE;
  const int lr = lane & 15, g4 = lane >> 4;

  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* ss = reinterpret_cast<float*>(smem);  // [Dp][17] state columns
  float* xs = ss + Dp * 17;                    // [64][17] V - exp(G) K S
  float* us = xs + 64 * 17;                    // [64][17] U
  float* uw = us + 64 * 17;                    // [64][17] exp(G_last - G) U

  const bool fresh = pos0[n_short + e] == 0;
  float* sg = state + ((long)slots[n_short + e] * H + h) * (long)D * V;
  for (int i = tid; i < Dp * 16; i += 256) {
    const int d = i >> 4, v = v0 + (i & 15);
    ss[d * 17 + (i & 15)] =
        (!fresh && d < D && v < V) ? sg[(long)d * V + v] : 0.0f;
  }
  __syncthreads();

  const long rstride = (long)KH * Dp;
  const f32x4 zero = {0, 0, 0, 0};
  const int row = wid * 16 + lr;            // A-operand row
  for (int c = chunk_cu[e]; c < chunk_cu[e + 1]; ++c) {
    const int i0 = chunks[2 * c] - tok_base;
    const int len = chunks[2 * c + 1];
    const long ch = (long)c * H + h;
    const float* kp = kn + ((long)i0 * KH + kh) * Dp;
    const float* qp = qn + ((long)i0 * KH + kh) * Dp;
    const float* tp = kt + ((long)i0 * KH + kh) * Dp;
    const float* gc = ge + ch * (CH ? Dp : 128);

    f32x4 ks = zero, qs = zero;
    {
      const float* ka = kp + row * rstride + g4 * 4;
      const float* qa = qp + row * rstride + g4 * 4;
      const bool in = row < len;
#pragma unroll 4
      for (int d = 0; d < Dp; d += 16) {
        const f32x4 a = in ? load4(ka + d) : zero;
        const f32x4 b = in ? load4(qa + d) : zero;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const float sv = ss[(d + g4 * 4 + s) * 17 + lr];
          ks = mma4(a[s], sv, ks);
          qs = mma4(b[s], sv, qs);
        }
      }
    }
    float gr[4], gl[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = wid * 16 + g4 * 4 + r;
      gr[r] = CH ? 1.0f : gc[i];
      gl[r] = CH ? 1.0f : gc[64 + i];
      const float v =
          i < len ? (float)vn[((long)(i0 + i) * H + h) * Vp + v0 + lr] : 0.0f;
      xs[i * 17 + lr] = v - gr[r] * ks[r];
    }
    __syncthreads();
    f32x4 u = zero;
    const float* ta = tm + ch * 4096 + row * 64 + g4 * 4;
    for (int j = 0; j <= wid; ++j) {
      const f32x4 a = load4(ta + j * 16);
#pragma unroll
      for (int s = 0; s < 4; ++s)
        u = mma4(a[s], xs[(j * 16 + g4 * 4 + s) * 17 + lr], u);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = wid * 16 + g4 * 4 + r;
      us[i * 17 + lr] = u[r];
      uw[i * 17 + lr] = u[r] * gl[r];
    }
    __syncthreads();
    f32x4 oc;
#pragma unroll
    for (int r = 0; r < 4; ++r) oc[r] = gr[r] * qs[r];
    const float* aa = am + ch * 4096 + row * 64 + g4 * 4;
    for (int j = 0; j <= wid; ++j) {
      const f32x4 a = load4(aa + j * 16);
#pragma unroll
      for (int s = 0; s < 4; ++s)
        oc = mma4(a[s], us[(j * 16 + g4 * 4 + s) * 17 + lr], oc);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = wid * 16 + g4 * 4 + r;
      if (i < len) o[((long)(i0 + i) * H + h) * Vp + v0 + lr] = oc[r];
    }
    for (int d0 = wid * 16; d0 < Dp; d0 += 64) {
      f32x4 sn;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sn[r] = gc[CH ? d0 + g4 * 4 + r : 63] * ss[(d0 + g4 * 4 + r) * 17 + lr];
      const float* ka = tp + d0 + lr;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int i = j * 16 + g4 * 4 + s;
          const float a = i < len ? ka[i * rstride] : 0.0f;
          sn = mma4(a, uw[i * 17 + lr], sn);
        }
#pragma unroll
      for (int r = 0; r < 4; ++r) ss[(d0 + g4 * 4 + r) * 17 + lr] = sn[r];
    }
    __syncthreads();
  }
  for (int i = tid; i < Dp * 16; i += 256) {
    const int d = i >> 4, v = v0 + (i & 15);
    if (d < D && v < V) sg[(long)d * V + v] = ss[d * 17 + (i & 15)];
  }
}

// The same walk with the state depth fixed at 32 * KD, CT column tiles a block, and
// eight waves: four for the state (K S, then U, then the next S), four for the outputs
// (Q S, A U); a SIMD has one of each, and both split K of the next chunk.  Chunks follow
// one another, so what counts is the way from one state to the next: three products with
// a barrier behind each.
//   * Every operand is a sum of three bf16 parts that keep all of its 24 bits, and a
//     product is that of eight pairs of parts: the ninth lies 2^-32 below the first.  The
//     matrix cores take 16 times as many bf16 products as fp32 ones, twice as many of
//     eight.  Sums of the largest pair and of the others are kept apart until the end.
//     Off by, in 2^-24 of the terms' magnitudes, at most (root of the mean square), fp32
//     and these: one term 1.00 (.42), 1.00 (.42); 8 terms 2.9 (.46), 2.0 (.24); 128 terms
//     3.9 (.47), .91 (.11); with six pairs a term alone is off by up to 2.7.  Numbers that
//     are not finite, or round up past the largest bf16 number, make NaN, where an fp32
//     product may be infinite.
//   * Parts of K lie in LDS, once for its rows (K S) and for its columns (the next S,
//     read transposed), split there a chunk ahead; pieces of a row are swapped by the
//     row, so that neither way of reading meets banks twice.
//   * S, U and what leads to U lie transposed in LDS, [column][row], parts apart.
//   * column blocks of one (request, head) read the same operands and run on one XCD;
//     two column tiles a block halve what comes out of its L2, where there are blocks
//     enough.
// CH: decays per channel; K for the state (kt) is another array, split in the chunk
// that it is for.
// Rows past the end of a chunk repeat its last one: their beta is 0, so they write
// nothing, and their outputs are not stored.
// Bound by what the two waves of a SIMD issue: of 8400 cycles a chunk (two tiles, depth
// 128) with six pairs 2900 are products, 3900 splits and what goes with them; with half of
// the products it takes 12% less, with splits left out 23%.  All of K by the output waves:
// 9700.
// Depth 128, 32 heads, fp32 products, six pairs, eight: 2 x 4001 tokens 371, 277, 303 us,
// 11 requests of 17 to 1160 374, 280, 303; decays per channel, 16 heads, 13 of 17 to 900
// 236, 183, 197; layers of 8 and 16 deep heads, padded to 32, 2 x 4001 tokens 233 to 221
// and 239 to 226 us.  Errors of a layer against 64 bits .88 to .96 of those of fp32.
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// eight numbers in three bf16 parts each, rounded: the third is exact
struct Parts8 {
  bf16x8 p[3];
};
// The next bf16 part of two numbers, cut off; else rounded.  Of a product one side is cut
// off and the other rounded: what is left out then has no sign of its own.
__device__ __forceinline__ unsigned cut_pair(float& x, float& y, bool more) {
  const unsigned a = __float_as_uint(x), b = __float_as_uint(y);
  if (more) {
    x -= __uint_as_float(a & 0xFFFF0000u);
    y -= __uint_as_float(b & 0xFFFF0000u);
  }
  return __builtin_amdgcn_perm(b, a, 0x07060302);
}
__device__ __forceinline__ unsigned round_pair(float& x, float& y, bool more) {
  const unsigned p = __builtin_bit_cast(unsigned, bf16x2{(__bf16)x, (__bf16)y});
  if (more) {
    x -= __uint_as_float(p << 16);
    y -= __uint_as_float(p & 0xFFFF0000u);
  }
  return p;
}
template <bool CUT, int N, typename V>
__device__ __forceinline__ void split3(float (&v)[N], V (&to)[3]) {
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    unsigned pairs[N / 2];
#pragma unroll
    for (int j = 0; j < N; j += 2)
      pairs[j / 2] = CUT ? cut_pair(v[j], v[j + 1], i < 2) : round_pair(v[j], v[j + 1], i < 2);
    to[i] = __builtin_bit_cast(V, pairs);
  }
}
__device__ __forceinline__ void split8(const f32x4& a, const f32x4& b, Parts8& to) {
  float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  split3<true>(v, to.p);
}

template <typename T, int KD, int CT, bool CH>
__global__ __launch_bounds__(512, 2) void delta_walk_fixed_kernel(
    const float* __restrict__ qn, const float* __restrict__ kn,
    const float* __restrict__ ktn, const T* __restrict__ vn, const float* __restrict__ tm,
    const float* __restrict__ am, const float* __restrict__ ge,
    float* __restrict__ state, float* __restrict__ o,
    const int* __restrict__ chunks, const int* __restrict__ chunk_cu,
    const int* __restrict__ pos0, const int* __restrict__ slots, int n_short,
    int tok_base, int n_long, int KH, int H, int D, int V, int Vp) {
  constexpr int Dp = KD * 32, ND = Dp / 16;
  constexpr int NT = (ND + 3) / 4;         // state row tiles per wave
  constexpr int KB = DR_CHUNK * Dp * 2;    // bytes of one part of a chunk of K
  constexpr int SB = CT * 16 * Dp * 2;     // ... of the state
  constexpr int UB = CT * 16 * DR_CHUNK * 2;  // ... of U
  const int cols = Vp / (16 * CT), pairs = H * n_long;
  int pair = blockIdx.x / cols, vt = blockIdx.x % cols;
  if (pairs % 8 == 0) {  // blocks go round the XCDs
    const int slot = blockIdx.x >> 3;
    pair = slot / cols * 8 + (blockIdx.x & 7);
    vt = slot % cols;
  }
  const int e = pair / H, h = pair % H;
  const int v0 = vt * 16 * CT;
  const int kh = h / (H / KH);
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int w = wid & 3;
  const int lr = lane & 15, g4 = lane >> 4;

  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* const kl = smem;              // [2][3][64][Dp] K by turns; CH: K, kt
  char* const st = kl + 6 * KB;       // [3][CT * 16][Dp] state
  char* const xt = st + 3 * SB;       // [3][CT * 16][64] V - exp(G) K S
  char* const ut = xt + 3 * UB;       // U
  char* const wt = ut + 3 * UB;       // exp(G_last - G) U (CH: U), tokens as K is read

  // byte of an element in rows of Dp, by pieces of 32 bytes, and in rows of 64 tokens, by
  // pieces of 16
  auto deep = [](int row, int d) {
    return row * Dp * 2 + (((d >> 4) ^ (row & (ND < 8 ? ND - 1 : 7))) << 5) + (d & 15) * 2;
  };
  auto wide = [](int col, int i) {
    return col * 128 + (((i >> 3) ^ (col & 7)) << 4) + (i & 7) * 2;
  };
  auto get8 = [](const char* p, int part, Parts8& to) {
#pragma unroll
    for (int i = 0; i < 3; ++i) to.p[i] = *reinterpret_cast<const bf16x8*>(p + i * part);
  };
  auto put4 = [](auto cut, const f32x4& x, char* p, int part) {
    float v[4] = {x[0], x[1], x[2], x[3]};
    bf16x4 to[3];
    split3<decltype(cut)::value>(v, to);
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x4*>(p + i * part) = to[i];
  };
  // a product of CT tiles; small: sums of all pairs of parts but the largest
  auto product = [](const Parts8& a, const Parts8 (&b)[CT], f32x4 (&sum)[CT],
                    f32x4 (&small)[CT]) {
    constexpr int I[8] = {1, 2, 0, 2, 1, 0, 0, 1}, J[8] = {2, 1, 2, 0, 1, 0, 1, 0};
#pragma unroll
    for (int q = 0; q < 8; ++q)
#pragma unroll
      for (int t = 0; t < CT; ++t) {
        f32x4& to = q == 5 ? sum[t] : small[t];
        to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.p[I[q]], b[t].p[J[q]], to, 0, 0, 0);
      }
  };

  // the two kinds of waves have loops of their own, with the same barriers
  auto walk = [&](auto kind) {
    constexpr bool keeps = decltype(kind)::value;  // a state wave
    const bool fresh = pos0[n_short + e] == 0;
    float* sg = state + ((long)slots[n_short + e] * H + h) * (long)D * V;
    const f32x4 zero = {0, 0, 0, 0};
    f32x4 own[NT][CT];                     // this wave's rows of the state
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int d0 = w * 16 + n * 64 + g4 * 4;
#pragma unroll
      for (int t = 0; t < CT; ++t) {
        const int v = v0 + t * 16 + lr;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          own[n][t][r] = keeps && !fresh && d0 + r < D && v < V
                             ? sg[(long)(d0 + r) * V + v] : 0.0f;
        if (keeps && d0 < Dp) put4(std::false_type{}, own[n][t], st + deep(t * 16 + lr, d0), SB);
      }
    }

    const int row = w * 16 + lr;              // A-operand row
    const int row_c = w * 16 + g4 * 4;        // first C row
    const unsigned vrow = H * Vp, krow = KH * Dp;  // from row to row
    // 0, unknown to the compiler: scalar loads come in any order, and a wait for LDS
    // would be one for all of them
    unsigned nought = 0;
    asm volatile("" : "+v"(nought));
    // what comes a chunk ahead: T or A, rows of Q and K (output waves), V and decays
    struct Ahead {
      f32x4 m[4], gr, gl, gd[NT], q[2 * KD], k[KD], kt[CH ? KD : 1];
      T v[CT][4];
      float all;
    };
    // what is above is asked for before what follows is begun
    auto issued = [] { __builtin_amdgcn_sched_barrier(0); };
    // a lane's pieces of 4 columns of this wave's 8 rows of K: a load takes whole lines
    constexpr int PR = Dp / 4;                // pieces of a row
    auto k_row = [&](int s) { return wid * 8 + s * (64 / PR) + lane / PR; };
    auto fetch_k = [&](const float* src, f32x4* to, int i0, int len) {
      const float* from = src + ((long)i0 * KH + kh) * Dp + lane % PR * 4;
#pragma unroll
      for (int s = 0; s < KD; ++s)
        to[s] = load4(from + (unsigned)min(k_row(s), len - 1) * krow);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto put_k = [&](const f32x4* k, char* to) {
      float v[4 * KD];
#pragma unroll
      for (int i = 0; i < 4 * KD; ++i) v[i] = k[i / 4][i % 4];
      // part by part: a wave alone would wait for each of its steps
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        unsigned pairs[2 * KD];
#pragma unroll
        for (int j = 0; j < 2 * KD; ++j) pairs[j] = cut_pair(v[2 * j], v[2 * j + 1], i < 2);
        issued();
#pragma unroll
        for (int s = 0; s < KD; ++s)
          *reinterpret_cast<uint2*>(to + i * KB + deep(k_row(s), lane % PR * 4)) =
              uint2{pairs[2 * s], pairs[2 * s + 1]};
      }
    };
    // What comes a chunk ahead is asked for piece by piece, between products: a wave that
    // asks for all at once waits for the loads before it (4400 cycles of 11700 a chunk).
    auto fetch_m = [&](Ahead& f, int c) {
      const long ch = (long)c * H + h;
      const float* mp = (keeps ? tm : am) + ch * 4096 + row * 64 + g4 * 8;
      f.m[0] = load4(mp);
      f.m[1] = load4(mp + 4);
      if (w >= 2) {
        f.m[2] = load4(mp + 32);
        f.m[3] = load4(mp + 36);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto fetch_g = [&](Ahead& f, int c) {
      const float* gc = ge + ((long)c * H + h) * (CH ? Dp : 128);
      if (!CH) f.gr = load4(gc + row_c);
      if constexpr (keeps) {
        if constexpr (!CH) {
          f.gl = load4(gc + 64 + row_c);
          f.all = gc[63 + nought];
        } else {
#pragma unroll
          for (int n = 0; n < NT; ++n) {
            const int d0 = w * 16 + n * 64;
            if (d0 < Dp) f.gd[n] = load4(gc + d0 + g4 * 4);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto fetch_v = [&](Ahead& f, int i0, int len, int t) {
      const T* vp = vn + ((long)i0 * H + h) * Vp + v0;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        f.v[t][r] = vp[(unsigned)min(row_c + r, len - 1) * vrow + (unsigned)(t * 16 + lr)];
      __builtin_amdgcn_sched_barrier(0);
    };
    auto fetch_q = [&](Ahead& f, int i0, int len, int d) {
      const float* qp = qn + ((long)i0 * KH + kh) * Dp + (unsigned)min(row, len - 1) * krow +
                        g4 * 8;
      f.q[2 * d] = load4(qp + d * 32);
      f.q[2 * d + 1] = load4(qp + d * 32 + 4);
      __builtin_amdgcn_sched_barrier(0);
    };
    // a barrier for what waves wrote into LDS; loads to registers go on
    auto sync_lds = [] {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };

    const int c_end = chunk_cu[e + 1];
    int c = chunk_cu[e];
    int i0 = chunks[2 * c] - tok_base, len = chunks[2 * c + 1];
    int cn = min(c + 1, c_end - 1);  // the last one is fetched twice
    int j0 = chunks[2 * cn] - tok_base, jl = chunks[2 * cn + 1];
    Ahead now = {};
    fetch_m(now, c);
    fetch_g(now, c);
    if constexpr (keeps) {
#pragma unroll
      for (int t = 0; t < CT; ++t) fetch_v(now, i0, len, t);
    } else {
#pragma unroll
      for (int d = 0; d < KD; ++d) fetch_q(now, i0, len, d);
    }
    fetch_k(kn, now.k, i0, len);
    if constexpr (CH) fetch_k(ktn, now.kt, i0, len);
    put_k(now.k, kl);
    __syncthreads();

    for (int buf = 0; c < c_end; ++c, buf ^= 1) {
      const int ahead = min(cn + 1, c_end - 1);
      const int* then = chunks + 2 * (ahead + nought);  // at any multiple of 4 bytes
      const int then_row = then[0], then_len = then[1];
      Ahead next = {};
      const char* k = kl + (CH ? 0 : buf * 3 * KB);
      const char* kt = kl + (CH ? 3 : buf * 3) * KB;

      f32x4 acc[CT], low[CT];
#pragma unroll
      for (int t = 0; t < CT; ++t) acc[t] = low[t] = zero;
      // Rows of K or Q times the state, 32 of the depth at a time.  Reads stand well ahead
      // of the products, and splitting between them.
      Parts8 ra[keeps ? 2 : 1], rb[2][CT];
      auto read = [&](int d) {
        if constexpr (keeps) get8(k + deep(row, d * 32 + g4 * 8), KB, ra[d & 1]);
#pragma unroll
        for (int t = 0; t < CT; ++t)
          get8(st + deep(t * 16 + lr, d * 32 + g4 * 8), SB, rb[d & 1][t]);
        issued();
      };
      auto rows_of = [&](int d) {
        if constexpr (keeps) {
          product(ra[d & 1], rb[d & 1], acc, low);
        } else {
          split8(now.q[2 * d], now.q[2 * d + 1], ra[0]);
          product(ra[0], rb[d & 1], acc, low);
        }
        issued();
      };
      // the matrix of this wave, whose tiles above the diagonal are not there
      Parts8 m[2];
      auto matrix = [&] {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const bool there = j * 2 + (g4 >> 1) <= w;
          split8(there ? now.m[2 * j] : zero, there ? now.m[2 * j + 1] : zero, m[j]);
        }
        issued();
      };
      // ... times columns of `x`; beside tiles that are not there, zeros, lie tokens of this
      // wave's own tile: what is no number in a later one stays there
      Parts8 lb[2][CT];
      auto read_lower = [&](const char* x) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int t = 0; t < CT; ++t)
            get8(x + wide(t * 16 + lr, min(j * 32 + g4 * 8, w * 16 + 8)), UB, lb[j][t]);
        issued();
      };
      auto lower = [&](f32x4 (&to)[CT], f32x4 (&small)[CT]) {
        product(m[0], lb[0], to, small);
        if (w >= 2) product(m[1], lb[1], to, small);
      };
      constexpr int HALF = (KD + 1) / 2;  // of the output waves' steps, in the first phase
      if constexpr (keeps) {
        read(0);
        if (KD > 1) read(1);
        float vf[CT][4];
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) vf[t][r] = (float)now.v[t][r];
        matrix();
#pragma unroll
        for (int d = 0; d < KD; ++d) {
          rows_of(d);
          if (d + 2 < KD) read(d + 2);
        }
        fetch_g(next, cn);
        fetch_k(kn, next.k, j0, jl);
        if constexpr (CH) put_k(now.kt, kl + 3 * KB);
#pragma unroll
        for (int t = 0; t < CT; ++t) {
          f32x4 x;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float s = acc[t][r] + low[t][r];
            x[r] = vf[t][r] - (CH ? s : now.gr[r] * s);
          }
          put4(std::false_type{}, x, xt + wide(t * 16 + lr, row_c), UB);
        }
      } else {
#pragma unroll
        for (int d = 0; d < HALF; ++d) read(d);
        if constexpr (CH) put_k(now.kt, kl + 3 * KB);
        fetch_g(next, cn);
        fetch_k(kn, next.k, j0, jl);
#pragma unroll
        for (int d = 0; d < HALF; ++d) rows_of(d);
      }
      sync_lds();

      // columns of kt: four tokens of one column out of rows, a lane's of 32 are
      // 4 g4 .. + 3 and 16 more
      Parts8 ka[NT][2];
      auto columns = [&] {
        const char* from = kt;
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const int d0 = min(w * 16 + n * 64, Dp - 16);
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int i = 0; i < 3; ++i) {
              s16x4 v[2];
#pragma unroll
              for (int q = 0; q < 2; ++q) {
                const int token = j * 32 + q * 16 + g4 * 4 + (lr >> 2);
                v[q] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) s16x4*)(
                        from + i * KB + deep(token, d0 + (lr & 3) * 4)));
              }
              ka[n][j].p[i] = __builtin_bit_cast(
                  bf16x8, __builtin_shufflevector(v[0], v[1], 0, 1, 2, 3, 4, 5, 6, 7));
            }
        }
      };
      // place of four tokens of a row as columns() has them
      const int turned = (w >> 1) * 32 + g4 * 8 + (w & 1) * 4;
      if constexpr (keeps) {
        f32x4 u[CT], small[CT];
#pragma unroll
        for (int t = 0; t < CT; ++t) u[t] = small[t] = zero;
        read_lower(xt);
        if (!CH) columns();
        issued();
        lower(u, small);
        fetch_m(next, cn);
        if constexpr (CH) fetch_k(ktn, next.kt, j0, jl);
#pragma unroll
        for (int t = 0; t < CT; ++t) {
#pragma unroll
          for (int r = 0; r < 4; ++r) u[t][r] += small[t][r];
          put4(std::false_type{}, u[t], ut + wide(t * 16 + lr, row_c), UB);
          if (!CH) {
#pragma unroll
            for (int r = 0; r < 4; ++r) u[t][r] *= now.gl[r];
          }
          put4(std::false_type{}, u[t], wt + wide(t * 16 + lr, turned), UB);
        }
      } else {
#pragma unroll
        for (int d = HALF; d < KD; ++d) read(d);
        matrix();
#pragma unroll
        for (int d = HALF; d < KD; ++d) rows_of(d);
        if constexpr (CH) fetch_k(ktn, next.kt, j0, jl);
#pragma unroll
        for (int d = 0; d < HALF; ++d) fetch_q(next, j0, jl, d);
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            acc[t][r] += low[t][r];
            low[t][r] = 0.0f;
            if (!CH) acc[t][r] *= now.gr[r];
          }
      }
      sync_lds();

      if constexpr (keeps) {
        if (CH) columns();
        Parts8 b[2][CT];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int t = 0; t < CT; ++t) get8(wt + wide(t * 16 + lr, j * 32 + g4 * 8), UB, b[j][t]);
        issued();
        f32x4 small[NT][CT];
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
          for (int t = 0; t < CT; ++t) {
            small[n][t] = zero;
#pragma unroll
            for (int r = 0; r < 4; ++r) own[n][t][r] *= CH ? now.gd[n][r] : now.all;
          }
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int n = 0; n < NT; ++n) product(ka[n][j], b[j], own[n], small[n]);
#pragma unroll
        for (int t = 0; t < CT; ++t) fetch_v(next, j0, jl, t);
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const int d0 = w * 16 + n * 64;
          if (d0 >= Dp) continue;
#pragma unroll
          for (int t = 0; t < CT; ++t) {
#pragma unroll
            for (int r = 0; r < 4; ++r) own[n][t][r] += small[n][t][r];
            put4(std::false_type{}, own[n][t], st + deep(t * 16 + lr, d0 + g4 * 4), SB);
          }
        }
        put_k(next.k, kl + (CH ? 0 : (buf ^ 1) * 3 * KB));
      } else {
        read_lower(ut);
        put_k(next.k, kl + (CH ? 0 : (buf ^ 1) * 3 * KB));
        issued();
        lower(acc, low);
        fetch_m(next, cn);
#pragma unroll
        for (int d = HALF; d < KD; ++d) fetch_q(next, j0, jl, d);
        float* op = o + ((long)i0 * H + h) * Vp + v0;
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (row_c + r < len)
              op[(unsigned)(row_c + r) * vrow + t * 16 + lr] = acc[t][r] + low[t][r];
      }
      sync_lds();
      now = next;
      i0 = j0;
      len = jl;
      cn = ahead;
      j0 = __builtin_amdgcn_readfirstlane(then_row) - tok_base;
      jl = __builtin_amdgcn_readfirstlane(then_len);
    }
    if (!keeps) return;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int d0 = w * 16 + n * 64 + g4 * 4;
#pragma unroll
      for (int t = 0; t < CT; ++t) {
        const int v = v0 + t * 16 + lr;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (d0 + r < D && v < V) sg[(long)(d0 + r) * V + v] = own[n][t][r];
      }
    }
  };
  if (wid < 4) {
    walk(std::true_type{});
  } else {
    walk(std::false_type{});
  }
}

// ---------------------------------------------------------------------------
// Step 4: output norm over V, weight, gate.  One wave per (token, head).
// ---------------------------------------------------------------------------

// NV groups of CW channels per lane, V <= 64 * CW * NV; DG_ROWS rows per wave
// in flight.
#define DG_ROWS 8

template <typename T, int NV, int CW>
__global__ __launch_bounds__(256) void delta_gate_kernel(
    const float* __restrict__ o, const T* __restrict__ z,
    const T* __restrict__ norm_w, T* __restrict__ out, long n, int tok_base,
    DeltaDims dm, int Vp, float eps) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const long w0 = ((long)blockIdx.x * 4 + wid) * DG_ROWS;
  const long rows = n * dm.H;
  float ov[DG_ROWS][NV][CW], gv[DG_ROWS][NV][CW];
#pragma unroll
  for (int k = 0; k < DG_ROWS; ++k) {
    const int wi = (int)min(w0 + k, rows - 1);
    const int i = wi / dm.H;
    const int h = wi - i * dm.H;
    const T* gr = z + (long)(tok_base + i) * dm.zstride + dm.gc + h * dm.V;
    const float* orow = o + (long)wi * Vp;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int v = min((lane + u * WAVE) * CW, dm.V - CW);
      load_lanes<float, CW>(orow + v, ov[k][u]);
      load_lanes<T, CW>(gr + v, gv[k][u]);
    }
  }
  float wv[NV][CW];
#pragma unroll
  for (int u = 0; u < NV; ++u)
    load_lanes<T, CW>(norm_w + min((lane + u * WAVE) * CW, dm.V - CW), wv[u]);
#pragma unroll
  for (int k = 0; k < DG_ROWS; ++k) {
    const long wi = w0 + k;
    if (wi >= rows) return;
    float ss = 0.0f;
#pragma unroll
    for (int u = 0; u < NV; ++u)
      if ((lane + u * WAVE) * CW < dm.V) {
#pragma unroll
        for (int q = 0; q < CW; ++q) ss += ov[k][u][q] * ov[k][u][q];
      }
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / (float)dm.V + eps);
    // row wi of [tokens * heads, V]
    T* dst = out + (tok_base * (long)dm.H + wi) * dm.V;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int v = (lane + u * WAVE) * CW;
      float r[CW];
#pragma unroll
      for (int q = 0; q < CW; ++q)
        r[q] = ov[k][u][q] * inv * wv[u][q] * out_gate(gv[k][u][q], dm.sigmoid);
      if (v < dm.V) store_lanes<T, CW>(dst + v, r);
    }
  }
}

struct DeltaLongArgs {
  const void *y, *z, *conv_w, *A_log, *dt_bias, *norm_w;
  float* state;
  void *conv_state, *out;
  float *qn, *kn, *lg, *bt, *tm, *am, *ge, *o, *qg, *kg, *kl;
  void* vn;
  const int *cu, *pos0, *slots, *tok_entry, *chunks, *chunk_cu;
  int n_short, n_long, tok_base, n_chunks, Dp, Vp;
  long n_tok;
  float eps;
};

template <typename T, int KD, int CT, bool CH>
static void delta_walk_tiles(const DeltaLongArgs& a, const DeltaDims& dm,
                             const float* q, const float* k, const float* kt,
                             int KH, hipStream_t stream) {
  // three parts of two bytes: K twice, the state, and X, U and W
  const int smem = 6 * (2 * DR_CHUNK * KD * 32 + CT * 16 * (KD * 32 + 3 * DR_CHUNK));
  if (smem > 65536)
    (void)hipFuncSetAttribute(
        reinterpret_cast<const void*>(&delta_walk_fixed_kernel<T, KD, CT, CH>),
        hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  const dim3 grid((unsigned)(a.Vp / (16 * CT) * dm.H * a.n_long));
  delta_walk_fixed_kernel<T, KD, CT, CH><<<grid, dim3(512), smem, stream>>>(
      q, k, kt, (const T*)a.vn, a.tm, a.am, a.ge, a.state, a.o, a.chunks,
      a.chunk_cu, a.pos0, a.slots, a.n_short, a.tok_base, a.n_long, KH, dm.H, dm.D,
      dm.V, a.Vp);
}

template <typename T, int KD, bool CH>
static void delta_walk_go(const DeltaLongArgs& a, const DeltaDims& dm,
                          const float* q, const float* k, const float* kt, int KH,
                          hipStream_t stream) {
  // A CU has one block, so with more than 256 column tiles two of them a block (a chunk of
  // two takes 1.3 times as long as of one).
  if (a.Vp % 32 == 0 && (long)a.Vp / 16 * dm.H * a.n_long > 256) {
    delta_walk_tiles<T, KD, 2, CH>(a, dm, q, k, kt, KH, stream);
  } else {
    delta_walk_tiles<T, KD, 1, CH>(a, dm, q, k, kt, KH, stream);
  }
}

// KH: heads that q, k and kt have
template <typename T, bool CH>
static void delta_walk_t(const DeltaLongArgs& a, const DeltaDims& dm,
                         const float* q, const float* k, const float* kt, int KH,
                         dim3 grid, hipStream_t stream) {
  const dim3 block(256);
#define DW_GO(N) delta_walk_go<T, N, CH>(a, dm, q, k, kt, KH, stream)
  if (a.Dp == 32) DW_GO(1);
  else if (a.Dp == 64) DW_GO(2);
  else if (a.Dp == 128) DW_GO(4);
  else {
    const size_t smem = ((size_t)a.Dp + 3 * 64) * 17 * sizeof(float);
    delta_walk_kernel<T, CH><<<grid, block, smem, stream>>>(
        q, k, kt, (const T*)a.vn, a.tm, a.am, a.ge, a.state, a.o, a.chunks,
        a.chunk_cu, a.pos0, a.slots, a.n_short, a.tok_base, KH, dm.H, dm.D,
        a.Dp, dm.V, a.Vp);
  }
#undef DW_GO
}

template <typename T>
static void delta_long_t(const DeltaLongArgs& a, const DeltaDims& dm,
                         hipStream_t stream) {
  const int C = 2 * dm.KH * dm.D + dm.H * dm.V;
  const float q_scale = 1.0f / sqrtf((float)dm.D);
  dim3 block(DC_BLOCK);
  // pairs of channels per lane where the sizes allow it
  const bool pair = dm.D % 2 == 0 && dm.V % 2 == 0 && dm.ystride % 2 == 0;
  const int cw = pair ? 2 : 1;
  const int pieces =
      2 * dm.KH + (dm.H * a.Vp + WAVE * cw - 1) / (WAVE * cw) + 1;
  const int groups = (pieces + DC_BLOCK / WAVE - 1) / (DC_BLOCK / WAVE);
  const dim3 g1((unsigned)((long)a.n_chunks * DC_SUB * groups));
#define DC_GO(N, W, TAPS)                                                    \
  delta_conv_kernel<T, N, W, TAPS><<<g1, block, 0, stream>>>(                \
      (const T*)a.y, (const T*)a.conv_w, (const T*)a.A_log,                  \
      (const T*)a.dt_bias, (const T*)a.conv_state, a.qn, a.kn, (T*)a.vn,     \
      a.lg, a.bt, a.cu, a.pos0, a.slots, a.tok_entry, a.chunks, a.tok_base,  \
      dm, a.Dp, a.Vp, q_scale, groups)
  if (pair) {
    if (a.Dp <= 128 && dm.taps == 4) DC_GO(1, 2, 4);
    else if (a.Dp <= 128) DC_GO(1, 2, DR_MAXTAPS);
    else if (a.Dp <= 256) DC_GO(2, 2, DR_MAXTAPS);
    else DC_GO(4, 2, DR_MAXTAPS);
  } else {
    if (a.Dp <= 64) DC_GO(1, 1, DR_MAXTAPS);
    else if (a.Dp <= 128) DC_GO(2, 1, DR_MAXTAPS);
    else if (a.Dp <= 256) DC_GO(4, 1, DR_MAXTAPS);
    else DC_GO(8, 1, DR_MAXTAPS);
  }
#undef DC_GO
  dim3 g2((unsigned)a.n_long, (unsigned)((C + DC_BLOCK - 1) / DC_BLOCK));
  if (dm.taps > 1)
    delta_conv_state_kernel<T><<<g2, block, 0, stream>>>(
        (const T*)a.y, (T*)a.conv_state, a.cu, a.pos0, a.slots, a.n_short, dm);
  dim3 g3((unsigned)a.n_chunks, (unsigned)dm.H);
  dim3 g4((unsigned)(a.Vp / 16), (unsigned)dm.H, (unsigned)a.n_long);
  if (dm.channels) {
    const bool vec = dm.D % 4 == 0 && dm.ac % 4 == 0 && dm.zstride % 4 == 0 &&
                     ((uintptr_t)a.z | (uintptr_t)a.dt_bias) % 16 == 0;
#define DCH_GO(V)                                                              \
  delta_chunk_channels_kernel<T, V><<<g3, block, 0, stream>>>(                 \
      a.qn, a.kn, (const T*)a.z, (const T*)a.A_log, (const T*)a.dt_bias, a.bt, \
      a.tm, a.am, a.qg, a.kg, a.kl, a.ge, a.chunks, a.tok_base, dm, a.Dp)
    if (vec) DCH_GO(true);
    else DCH_GO(false);
#undef DCH_GO
    delta_walk_t<T, true>(a, dm, a.qg, a.kg, a.kl, dm.H, g4, stream);
  } else {
    const long pairs = (long)a.n_chunks * dm.KH;
    const int r = dm.H / dm.KH;
    const int per = r % DC_HEADS == 0 && pairs * r >= 256 ? DC_HEADS : 1;
    const dim3 g((unsigned)((pairs + 7) / 8 * 8 * (r / per)));
    delta_chunk_kernel<<<g, block, 0, stream>>>(
        a.qn, a.kn, a.lg, a.bt, a.tm, a.am, a.ge, a.chunks, a.n_chunks, a.tok_base,
        dm.KH, dm.H, a.Dp, per);
    delta_walk_t<T, false>(a, dm, a.qn, a.kn, a.kn, dm.KH, g4, stream);
  }
  dim3 g5((unsigned)((a.n_tok * dm.H + 4 * DG_ROWS - 1) / (4 * DG_ROWS)));
#define DG_GO(N, W)                                                          \
  delta_gate_kernel<T, N, W><<<g5, block, 0, stream>>>(                      \
      a.o, (const T*)a.z, (const T*)a.norm_w, (T*)a.out, a.n_tok,            \
      a.tok_base, dm, a.Vp, a.eps)
  if (pair && dm.gc % 2 == 0 && dm.zstride % 2 == 0) {
    if (dm.V <= 128) DG_GO(1, 2);
    else if (dm.V <= 256) DG_GO(2, 2);
    else DG_GO(4, 2);
  } else {
    if (dm.V <= 64) DG_GO(1, 1);
    else if (dm.V <= 128) DG_GO(2, 1);
    else if (dm.V <= 256) DG_GO(4, 1);
    else DG_GO(8, 1);
  }
#undef DG_GO
}

extern "C" void launch_delta_long(const DeltaLongArgs* a, const DeltaDims* dm,
                                  bool f32, hipStream_t stream) {
  if (f32)
    delta_long_t<float>(*a, *dm, stream);
  else
    delta_long_t<__bf16>(*a, *dm, stream);
}
