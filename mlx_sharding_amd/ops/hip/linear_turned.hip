// q, k and v of few tokens: their product with the rows' norm, the rotations of queries and keys,
// and keys and values to the cache, up to 384 rows in one kernel.
//
// A tile of linear_own_kernel has the two dimensions that a rotation takes in one lane (row_of),
// which turns them as rounded, so that the results are those of the product and rope_qkv_kernel.
// That kernel is launch alone (57 rows of 2048, 32 + 4 + 4 heads of 64: product 7.4 us and turns
// 4.0, here 8.0; a prompt of three layers of them 147.8 -> 137.5 us).
#include "linear_turned.h"

#include "linear_own_kernel.h"

namespace {

struct TurnedRun {
  LinearFewArgs a;
  TurnedArgs t;
};

template <int RT, int TT>
__global__ __launch_bounds__(OWN_WAVES * WAVE) void linear_turned_kernel(const TurnedRun b) {
  const LinearFewArgs& a = b.a;
  const TurnedArgs& r = b.t;
  own_block<RT, TT, 1, TURNED_ROWS, true, false, false>(
      a, blockIdx.x, [&](int row, int col0, int lg, const f32x4& v, const Ends<0>&) {
        const int col = col0 + lg * 2;
        if (col >= a.O) return;
        const int half = a.n_zero, d = col & (half - 1), h = (col - d) / half;
        const int seq = row / r.T, t = row - seq * r.T;
        bf16x2_t u, w;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          float f = v[j], g = v[j + 2];
          if (a.bias) {
            f += (float)a.bias[h * 2 * half + d + j];
            g += (float)a.bias[h * 2 * half + d + j + half];
          }
          u[j] = (__bf16)f, w[j] = (__bf16)g;
        }
        if (h < r.Hq + r.Hkv) {
          const float* c = r.cos + t * half + d;
          const float* s = r.sin + t * half + d;
          bf16x2_t y, z;
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            y[j] = (__bf16)((float)u[j] * c[j] - (float)w[j] * s[j]);
            z[j] = (__bf16)((float)w[j] * c[j] + (float)u[j] * s[j]);
          }
          u = y, w = z;
        }
        __bf16* to;
        if (h < r.Hq) {
          to = a.y + ((long)row * r.Hq + h) * 2 * half + d;
        } else {
          const bool key = h < r.Hq + r.Hkv;
          const long head = (long)seq * r.Hkv + h - r.Hq - (key ? 0 : r.Hkv);
          to = (key ? r.kcache : r.vcache) + (head * r.cap + r.at + t) * 2 * half + d;
        }
        *reinterpret_cast<bf16x2_t*>(to) = u;
        *reinterpret_cast<bf16x2_t*>(to + half) = w;
      });
}

}  // namespace

extern "C" bool linear_turned_takes(long M, long heads, long D, long K) {
  return M >= 1 && M <= 384 && K >= 32 && K % 32 == 0 && K <= 32768 && D >= 32 && D <= 256 &&
         (D & (D - 1)) == 0 && heads * D < 1L << 24 &&
         tiles_beside((int)M, (int)(heads * D / 16), 0, (int)K, true).rt > 0;
}

extern "C" void launch_linear_turned(const void* x, const void* w, const void* bias,
                                     const void* norm, void* q, int M, int K, int D, long ldx,
                                     long ldw, float eps, float offset, const TurnedArgs* t,
                                     hipStream_t stream) {
  TurnedRun b{};
  LinearFewArgs& a = b.a;
  b.t = *t;
  a.x = (const __bf16*)x, a.w = (const __bf16*)w, a.bias = (const __bf16*)bias;
  a.norm = (const __bf16*)norm, a.y = (__bf16*)q;
  a.M = (short)M, a.O = (t->Hq + 2 * t->Hkv) * D / 2, a.K = K, a.n_zero = D / 2;
  a.ldx = ldx, a.ldw = ldw, a.eps = eps, a.offset = offset;
  turned(a, LF_PLAIN, 64);
  const Tiles n = tiles_beside(M, a.O / 8, 0, K, true);
  with_tiles(n, [&](auto rt, auto tt) {
    const auto kernel = &linear_turned_kernel<rt(), tt()>;
    const int smem = own_room(n.rt, n.tt, 1, K, true);
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    kernel<<<n.blocks, OWN_WAVES * WAVE, smem, stream>>>(b);
  });
}
