// Python bindings for the gfx950 kernel library (torch extension).
// Pure HIP tree — no CUDA shims; built by hipcc via torch cpp_extension
// with PYTORCH_ROCM_ARCH=gfx950.

#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

#include "hip_common.h"
#include "linear_few.h"
#include "mla_decode.h"
#include "moe_rows.h"
#include "linear_turned.h"
#include "warm.h"
#include "moe_tiles.h"

extern "C" {
void launch_rms_norm(const void*, void*, const void*, long, int, float, float,
                     long, hipStream_t);
void launch_rms_norm_residual(const void*, const void*, void*, void*,
                              const void*, long, int, float, float,
                              hipStream_t);
void launch_norm_add(const void*, const void*, const void*, const void*, void*, void*,
                     long, int, float, float, float, float, hipStream_t);
void launch_glu(const void*, const void*, void*, long, bool, hipStream_t);
void launch_glu_strided(const void*, const void*, void*, long, int, long,
                        long, bool, hipStream_t);
void launch_softcap(const void*, void*, long, float, hipStream_t);
void launch_rope(const void*, void*, const float*, const float*, long, int,
                 int, int, bool, long, long, hipStream_t);
void launch_mla_append_kv(const void*, const void*, void*, void*, const int*,
                          int, int, int, int, int, int, int, long, long,
                          hipStream_t);
void launch_rope_qkv(const void*, const void*, const void*, const float*, const float*,
                     void*, void*, void*, const int*, long, long, int, int, int, int,
                     long, long, long, long, hipStream_t);
void launch_step_begin(const long*, const void*, const void*, const int*, const float*,
                       const float*, void*, float*, float*, long, long, int, long, int,
                       hipStream_t);
void launch_step_end(const void*, long, float*, int, int, int*, hipStream_t);
void launch_rope_append_kv(const void*, const void*, const float*,
                           const float*, void*, void*, const int*, int, int,
                           int, int, int, long, bool, long, long,
                           hipStream_t);
void launch_attn_decode(const void*, const void*, const void*, void*, float*,
                        float*, int, const int*, int, int, int, int, long,
                        int, int, long, float, float, int, hipStream_t);
bool attn_decode_supported_shape(int, int);
int attn_decode_tile(int, int, int, bool);
void launch_attn_decode_tile(const void*, const void*, const void*, void*,
                             float*, float*, int, const int*, int, int, int,
                             int, long, int, int, bool, bool, float, float, int,
                             hipStream_t);
bool attn_decode_wave(int, long, long);
void launch_attn_step(const void*, const void*, const void*, long, long, long,
                      const float*, const float*, void*, void*, void*, float*, float*,
                      unsigned*, int, const int*, int, int, int, int, long, int, float,
                      float, int, const Warm*, hipStream_t);
void launch_attn_prefill(const void*, const void*, const void*, void*, int,
                         int, int, int, int, long, long, long, long, long, int,
                         int, float, float, int, int, hipStream_t);
bool attn_prefill_supported(int, int);
void launch_latent_prompt(const void*, const void*, const void*, const void*, void*,
                          const int*, const int*, const int*, const int*, int, int, int,
                          int, long, int, float, hipStream_t);
void launch_mla_prompt(const void*, const void*, const void*, const float*,
                       const float*, void*, int, int, int, int, long, long, long, long,
                       int, float, int, hipStream_t);
void launch_mfma_probe(const void*, const void*, float*, hipStream_t);
void launch_w4a16_gemv(const void*, const void*, const void*, const void*,
                       void*, int, int, int, int, int, hipStream_t);
int w4a16_mfma_nsplit(int, int, int);
void launch_bf16_gemv_mfma(const void*, const void*, void*, float*, int, int,
                           int, int, hipStream_t);
int bf16_gemv_nsplit(int, int, int);
void launch_bf16_gemm_m64(const void*, const void*, void*, float*, int, int,
                          int, int, hipStream_t);
int bf16_gemm_m64_nsplit(int, int, int);
void launch_w4a16_mfma(const void*, const void*, const void*, const void*,
                       void*, float*, int, int, int, int, int, int,
                       hipStream_t);
void launch_dequant(const void*, const void*, const void*, void*, long, int,
                    int, int, hipStream_t);
void launch_moe_scatter_rows(const void*, void*, const int*, const int*, int,
                             int, hipStream_t);
void launch_moe_gather_reduce(const void*, const int*, const float*, const void*,
                              const void*, void*, int, int, int, hipStream_t);
void launch_moe_gateup_mfma(const void*, const void*, const void*, void*,
                            const int*, const int*, const int*, const int*,
                            int, int, int, hipStream_t);
void launch_moe_down_mfma(const void*, const void*, float*, const int*,
                          const int*, const int*, const int*, const float*,
                          int, int, int, hipStream_t);
void launch_moe_gateup_grouped(const void*, const void*, const void*, void*,
                               const int*, const int*, const int*, const int*,
                               int, int, int, hipStream_t);
void launch_moe_down_grouped(const void*, const void*, float*, const int*,
                             const int*, const int*, const int*, const float*,
                             int, int, int, hipStream_t);
void launch_moe_w4_mfma(const void*, const void*, const void*, const void*,
                        void*, const int*, const int*, const int*,
                        const int*, int, int, int, int, int, hipStream_t);
void launch_moe_gate_subranges(const void*, int*, float*, int*, int*, int*,
                               int, int, int, int, int, float, int,
                               hipStream_t);
void launch_moe_w4f16_gateup(const void*, const void*, const void*,
                             const void*, const void*, const void*,
                             const void*, void*, const int*, const int*,
                             const int*, const int*, int, int, int, int, int,
                             hipStream_t);
void launch_moe_w4f16_down(const void*, const void*, const void*, const void*,
                           float*, const int*, const int*, const int*,
                           const int*, const float*, int, int, int, int, int,
                           hipStream_t);
void launch_w4f16_gemv(const void*, const void*, const void*, const void*,
                       void*, float*, int, int, int, int, int, int,
                       hipStream_t);
int w4f16_gemv_nsplit(int, int, int);
void launch_gemm_kseg(const void*, const void*, void*, void*, int, int, int,
                      int, hipStream_t);
void launch_gemm_kseg_w4(const void*, const void*, const void*, const void*,
                         void*, void*, int, int, int, int, int, hipStream_t);
}

namespace {

hipStream_t cur_stream() {
  return c10::hip::getCurrentHIPStream().stream();
}

void check_bf16(const torch::Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda(), name, " must be on GPU");
  TORCH_CHECK(t.scalar_type() == torch::kBFloat16, name, " must be bf16");
}

// View t as [rows, last-dim] with a uniform row stride (a fused-output
// column-slice view qualifies) — lets kernels read split views in place
// instead of the binding materializing a .contiguous() copy per call.
bool row_view2(const torch::Tensor& t, long& rows, long& rstride) {
  const int d = t.dim();
  if (d < 2 || t.stride(d - 1) != 1) return false;
  if (d == 2) {
    rows = t.size(0);
    rstride = t.stride(0);
    return true;
  }
  if (d == 3) {
    if (t.stride(0) != t.size(1) * t.stride(1)) return false;
    rows = t.size(0) * t.size(1);
    rstride = t.stride(1);
    return true;
  }
  return false;
}

torch::Tensor rms_norm(torch::Tensor x, torch::Tensor w, double eps,
                       double w_off) {
  check_bf16(x, "x");
  check_bf16(w, "w");
  const int H = x.size(-1);
  TORCH_CHECK(H % 4 == 0, "H must be divisible by 4");
  long rows, rstride;
  torch::Tensor xv = x;
  if (!row_view2(x, rows, rstride) || rstride % 4 != 0
      || ((uintptr_t)x.data_ptr()) % 8 != 0) {  // short4v-aligned rows
    xv = x.contiguous();
    rows = xv.numel() / H;
    rstride = H;
  }
  auto y = torch::empty(x.sizes(), x.options());
  launch_rms_norm(xv.data_ptr(), y.data_ptr(), w.contiguous().data_ptr(), rows,
                  H, (float)eps, (float)w_off, rstride, cur_stream());
  return y;
}

std::vector<torch::Tensor> rms_norm_residual(torch::Tensor x,
                                             torch::Tensor resid,
                                             torch::Tensor w, double eps,
                                             double w_off) {
  check_bf16(x, "x");
  auto xc = x.contiguous();
  auto rc = resid.contiguous();
  const int H = xc.size(-1);
  long rows = xc.numel() / H;
  auto y = torch::empty_like(xc);
  auto h = torch::empty_like(xc);
  launch_rms_norm_residual(xc.data_ptr(), rc.data_ptr(), y.data_ptr(),
                           h.data_ptr(), w.contiguous().data_ptr(), rows, H,
                           (float)eps, (float)w_off, cur_stream());
  return {y, h};
}

// (residual + norm(x), with a next norm's weight its rows of that)
std::vector<torch::Tensor> norm_add(torch::Tensor x, torch::Tensor w, double eps,
                                    double off, torch::Tensor resid,
                                    c10::optional<torch::Tensor> w2, double eps2,
                                    double off2) {
  const long H = x.dim() ? x.size(-1) : 0;
  TORCH_CHECK(H >= 8 && H <= 8192 && H % 8 == 0 && x.numel() >= H, "row size");
  auto ok = [](const torch::Tensor& t, long n) {
    check_bf16(t, "operand");
    TORCH_CHECK(t.is_contiguous() && t.numel() == n &&
                    reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0, "layout");
  };
  ok(x, x.numel());
  ok(resid, x.numel());
  ok(w, H);
  if (w2.has_value()) ok(*w2, H);
  auto h = torch::empty_like(x);
  std::vector<torch::Tensor> out{h};
  if (w2.has_value()) out.push_back(torch::empty_like(x));
  launch_norm_add(x.data_ptr(), resid.data_ptr(), w.data_ptr(),
                  w2.has_value() ? w2->data_ptr() : nullptr, h.data_ptr(),
                  out.back().data_ptr(), x.numel() / H, (int)H, (float)eps,
                  (float)off, (float)eps2, (float)off2, cur_stream());
  return out;
}

torch::Tensor glu(torch::Tensor gate, torch::Tensor up, bool gelu) {
  check_bf16(gate, "gate");
  TORCH_CHECK(gate.numel() == up.numel(), "gate/up size mismatch");
  TORCH_CHECK(gate.numel() % 4 == 0, "numel must be divisible by 4");
  const int I = gate.size(-1);
  long growz, gstride, urows, ustride;
  // fused gate|up split views read in place (no .contiguous() copies)
  if (!(gate.is_contiguous() && up.is_contiguous())
      && row_view2(gate, growz, gstride) && row_view2(up, urows, ustride)
      && growz == urows && up.size(-1) == I && I % 4 == 0
      && gstride % 4 == 0 && ustride % 4 == 0
      && ((uintptr_t)gate.data_ptr()) % 8 == 0
      && ((uintptr_t)up.data_ptr()) % 8 == 0) {
    auto y = torch::empty(gate.sizes(), gate.options());
    launch_glu_strided(gate.data_ptr(), up.data_ptr(), y.data_ptr(), growz, I,
                       gstride, ustride, gelu, cur_stream());
    return y;
  }
  auto g = gate.contiguous();
  auto u = up.contiguous();
  auto y = torch::empty_like(g);
  launch_glu(g.data_ptr(), u.data_ptr(), y.data_ptr(), g.numel(), gelu,
             cur_stream());
  return y;
}

torch::Tensor softcap_op(torch::Tensor x, double cap) {
  check_bf16(x, "x");
  auto xc = x.contiguous();
  TORCH_CHECK(xc.numel() % 4 == 0, "numel must be divisible by 4");
  auto y = torch::empty_like(xc);
  launch_softcap(xc.data_ptr(), y.data_ptr(), xc.numel(), (float)cap,
                 cur_stream());
  return y;
}

// x: [B, T, nH, D]; cos/sin: [T, D/2] fp32
torch::Tensor apply_rope(torch::Tensor x, torch::Tensor cos, torch::Tensor sin,
                         bool interleaved) {
  check_bf16(x, "x");
  TORCH_CHECK(x.dim() == 4, "x must be [B, T, nH, D]");
  auto cc = cos.contiguous();
  auto sc = sin.contiguous();
  TORCH_CHECK(cc.scalar_type() == torch::kFloat32, "cos must be fp32");
  const int B = x.size(0), T = x.size(1), nH = x.size(2), D = x.size(3);
  TORCH_CHECK(cc.size(0) == T && cc.size(1) == D / 2, "cos shape mismatch");
  // fused-qkv splits / nope-rope slices read in place
  torch::Tensor xv = x;
  long rstride = (long)nH * D, hstride = D;
  const bool strided_ok = x.stride(3) == 1
      && x.stride(0) == x.size(1) * x.stride(1);
  if (strided_ok) {
    rstride = x.stride(1);
    hstride = x.stride(2);
  } else {
    xv = x.contiguous();
  }
  auto y = torch::empty({B, T, nH, D}, x.options());
  launch_rope(xv.data_ptr(), y.data_ptr(), cc.data_ptr<float>(),
              sc.data_ptr<float>(), (long)B * T, T, nH, D, interleaved,
              rstride, hstride, cur_stream());
  return y;
}

// q, k, v [B, T, heads, D], heads side by side; caches [B, Hkv, cap, D].  Returns the
// turned queries; keys (turned) and values go to the caches from row pos (pos0) on.
torch::Tensor rope_qkv(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                       torch::Tensor cos, torch::Tensor sin, torch::Tensor kcache,
                       torch::Tensor vcache, c10::optional<torch::Tensor> pos,
                       int64_t pos0) {
  const long B = q.size(0), T = q.size(1), D = q.size(3), Hkv = k.size(2);
  auto whole = [](const torch::Tensor& t) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  // from one token to the next
  auto row = [&](const torch::Tensor& t) { return t.stride(T == 1 ? 0 : 1); };
  for (const auto& t : {q, k, v}) {
    check_bf16(t, "operand");
    TORCH_CHECK(t.dim() == 4 && t.size(0) == B && t.size(1) == T && t.size(3) == D &&
                    t.stride(3) == 1 && t.stride(2) == D && row(t) % 8 == 0 &&
                    (B == 1 || T == 1 || t.stride(0) == T * row(t)) && whole(t), "rows");
  }
  TORCH_CHECK(D >= 16 && D % 16 == 0 && B >= 1 && T >= 1 && v.size(2) == Hkv &&
                  (q.size(2) + 3 * Hkv) * D < (1L << 30), "sizes");
  for (const auto& t : {kcache, vcache}) {
    check_bf16(t, "cache");
    TORCH_CHECK(t.dim() == 4 && t.size(0) == B && t.size(1) == Hkv &&
                    t.size(2) == kcache.size(2) && t.size(3) == D &&
                    t.is_contiguous() && whole(t), "caches");
  }
  for (const auto& t : {cos, sin})
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kFloat32 &&
                    t.is_contiguous() && t.numel() == T * D / 2, "rotations");
  const int* pp = nullptr;
  if (pos.has_value()) {
    TORCH_CHECK(pos->is_cuda() && pos->scalar_type() == torch::kInt32, "pos int32");
    pp = pos->data_ptr<int>();
  } else {
    TORCH_CHECK(pos0 >= 0 && pos0 + T <= kcache.size(2), "no room in the cache");
  }
  auto out = torch::empty({B, T, q.size(2), D}, q.options());
  launch_rope_qkv(q.data_ptr(), k.data_ptr(), v.data_ptr(), cos.data_ptr<float>(),
                  sin.data_ptr<float>(), out.data_ptr(), kcache.data_ptr(),
                  vcache.data_ptr(), pp, pos0, B * T, (int)T, (int)q.size(2), (int)Hkv,
                  (int)D, kcache.size(2), row(q), row(k), row(v),
                  cur_stream());
  return out;
}

static void check_position(const torch::Tensor& pos) {
  TORCH_CHECK(pos.is_cuda() && pos.scalar_type() == torch::kInt32 && pos.numel() == 1,
              "one int32 position");
}

// The embedding rows of tokens [...] (times scale), and row pos of cos and sin.
std::vector<torch::Tensor> step_begin(torch::Tensor tokens, torch::Tensor table,
                                      c10::optional<torch::Tensor> scale,
                                      torch::Tensor pos, torch::Tensor cos,
                                      torch::Tensor sin) {
  check_bf16(table, "embedding");
  TORCH_CHECK(tokens.is_cuda() && tokens.scalar_type() == torch::kInt64 &&
                  tokens.is_contiguous() && tokens.numel() >= 1, "tokens int64");
  TORCH_CHECK(table.dim() == 2 && table.is_contiguous() && table.size(0) >= 1 &&
                  table.size(1) >= 8 && table.size(1) % 8 == 0 &&
                  reinterpret_cast<uintptr_t>(table.data_ptr()) % 16 == 0, "embedding");
  if (scale.has_value()) {
    check_bf16(*scale, "scale");
    TORCH_CHECK(scale->numel() == 1, "one scale");
  }
  check_position(pos);
  for (const auto& t : {cos, sin})
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kFloat32 && t.dim() == 2 &&
                    t.is_contiguous() && t.sizes() == cos.sizes() && t.numel() >= 1,
                "tables of rotations");
  const long W = table.size(1), half = cos.size(1);
  TORCH_CHECK(tokens.numel() * (W / 8) < (1L << 32), "sizes");
  auto shape = tokens.sizes().vec();
  shape.push_back(W);
  auto h = torch::empty(shape, table.options());
  auto c = torch::empty({1, half}, cos.options()), s = torch::empty({1, half}, cos.options());
  launch_step_begin(tokens.data_ptr<long>(), table.data_ptr(),
                    scale.has_value() ? scale->data_ptr() : nullptr, pos.data_ptr<int>(),
                    cos.data_ptr<float>(), sin.data_ptr<float>(), h.data_ptr(),
                    c.data_ptr<float>(), s.data_ptr<float>(), tokens.numel(),
                    table.size(0), (int)W, cos.size(0), (int)half, cur_stream());
  return {h, c, s};
}

// x [rows, n] in fp32; the position moves on.
torch::Tensor step_end(torch::Tensor x, torch::Tensor pos) {
  check_bf16(x, "logits");
  check_position(pos);
  TORCH_CHECK(x.dim() == 2 && x.stride(1) == 1 && x.size(0) >= 1 && x.size(0) < 65536 &&
                  x.size(1) >= 1 && x.size(1) < (1L << 31) - 1024, "rows of logits");
  auto y = torch::empty(x.sizes(), x.options().dtype(torch::kFloat32));
  launch_step_end(x.data_ptr(), x.stride(0), y.data_ptr<float>(), (int)x.size(0),
                  (int)x.size(1), pos.data_ptr<int>(), cur_stream());
  return y;
}

// k/v [B, T, Hkv, D]; caches full buffers [B, Hkv, Scap, D]
void rope_append_kv(torch::Tensor k, torch::Tensor v, torch::Tensor cos,
                    torch::Tensor sin, torch::Tensor kcache,
                    torch::Tensor vcache, c10::optional<torch::Tensor> pos,
                    int64_t pos0, bool interleaved) {
  check_bf16(k, "k");
  TORCH_CHECK(k.dim() == 4, "k must be [B, T, Hkv, D]");
  auto cc = cos.contiguous();
  auto sc = sin.contiguous();
  TORCH_CHECK(cc.scalar_type() == torch::kFloat32, "cos must be fp32");
  const int B = k.size(0), T = k.size(1), Hkv = k.size(2), D = k.size(3);
  TORCH_CHECK(D % 2 == 0, "head dim must be even");
  TORCH_CHECK(cc.size(0) == T && cc.size(1) == D / 2, "cos shape mismatch");
  TORCH_CHECK(kcache.is_contiguous() && vcache.is_contiguous(),
              "caches contiguous");
  TORCH_CHECK(kcache.size(3) == D && vcache.size(3) == D, "cache D mismatch");
  const long Scap = kcache.size(2);
  const int* pp = nullptr;
  if (pos.has_value()) pp = pos->data_ptr<int>();
  // fused-qkv split views read in place (heads contiguous within slice)
  auto view_ok = [&](const torch::Tensor& t) {
    return t.stride(3) == 1 && t.stride(2) == D
        && t.stride(0) == t.size(1) * t.stride(1);
  };
  torch::Tensor kv = k, vv = v;
  long krs = (long)Hkv * D, vrs = (long)Hkv * D;
  if (view_ok(k)) krs = k.stride(1); else kv = k.contiguous();
  if (view_ok(v)) vrs = v.stride(1); else vv = v.contiguous();
  launch_rope_append_kv(kv.data_ptr(), vv.data_ptr(), cc.data_ptr<float>(),
                        sc.data_ptr<float>(), kcache.data_ptr(),
                        vcache.data_ptr(), pp, (int)pos0, B, T, Hkv, D, Scap,
                        interleaved, krs, vrs, cur_stream());
}

// kvh [B, T, nh, nope+vd]; kpe [B, T, rope]; caches full buffers
void mla_append_kv(torch::Tensor kvh, torch::Tensor kpe, torch::Tensor kcache,
                   torch::Tensor vcache, c10::optional<torch::Tensor> pos,
                   int64_t pos0) {
  check_bf16(kvh, "kvh");
  const int B = kvh.size(0), T = kvh.size(1), nh = kvh.size(2);
  const int rope = kpe.size(-1);
  const int kd = kcache.size(3);
  const int vd = vcache.size(3);
  const int nope = kd - rope;
  TORCH_CHECK(kvh.size(3) == nope + vd, "kvh dim mismatch");
  TORCH_CHECK(kcache.is_contiguous() && vcache.is_contiguous(), "caches contiguous");
  const long Scap = kcache.size(2);
  const int* pp = nullptr;
  if (pos.has_value()) pp = pos->data_ptr<int>();
  long kpe_rows, kpe_rs;
  torch::Tensor kpev = kpe;
  if (!row_view2(kpe, kpe_rows, kpe_rs)) {
    kpev = kpe.contiguous();
    kpe_rs = rope;
  }
  launch_mla_append_kv(kvh.contiguous().data_ptr(), kpev.data_ptr(),
                       kcache.data_ptr(), vcache.data_ptr(), pp, (int)pos0, B,
                       T, nh, nope, vd, rope, Scap, kpe_rs, cur_stream());
}

// Slices of the keys for the tile kernel: up to 512 blocks, two a CU, which are
// all at work at once, and no slice under one tile.  256 blocks leave half of the
// loads in flight unused (5 sequences of 5004 keys, 8 heads of 256: 68 us, 45 with
// 512), 1024 come in two rounds and double what the merge reads (48 us; 64 cached
// latents of 2048 tokens: 49 us, 40 with 512).  Whole steps of heads of 256 have one a CU.
static int decode_slices(long pairs, long span, int tile, int blocks = 512) {
  return (int)std::max<long>(
      1, std::min<long>({64, blocks / std::max<long>(pairs, 1),
                         (span + tile - 1) / tile}));
}

// q [B, Hq, 1, Dk]; k/v: cache views [B, Hkv, S, D] with row-contiguous
// last dim over a [B, Hkv, Scap, D] buffer.
torch::Tensor attn_decode(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                          double scale, double softcap, int64_t window,
                          c10::optional<torch::Tensor> pos) {
  check_bf16(q, "q");
  check_bf16(k, "k");
  TORCH_CHECK(q.size(2) == 1, "attn_decode needs Tq == 1");
  auto qc = q.contiguous();
  const int B = qc.size(0), Hq = qc.size(1), Dk = qc.size(3);
  const int Hkv = k.size(1), S = k.size(2);
  const int Dv = v.size(3);
  TORCH_CHECK(k.stride(3) == 1 && v.stride(3) == 1, "K/V rows must be contiguous");
  TORCH_CHECK(k.stride(2) == Dk, "K seq stride mismatch");
  // V rows may live inside the K rows (absorbed MLA: V = K[..., :Dv])
  const long vstride = v.stride(2);
  TORCH_CHECK(vstride >= Dv, "V seq stride too small");
  TORCH_CHECK(Hq % Hkv == 0, "Hq must be divisible by Hkv");
  TORCH_CHECK(Dk % 8 == 0, "Dk must be a multiple of 8");
  TORCH_CHECK(attn_decode_supported_shape(Hq / Hkv, Dv),
              "unsupported GQA ratio/Dv ", Hq / Hkv, " ", Dv);
  TORCH_CHECK(Dv <= 512, "Dv too large");
  long kScap = k.stride(1) / Dk;
  long vScap = v.stride(1) / vstride;
  TORCH_CHECK(kScap == vScap, "K/V capacity mismatch");
  auto out = torch::empty({B, Hq, 1, Dv}, qc.options());
  const int* s_ptr = nullptr;
  if (pos.has_value()) {
    TORCH_CHECK(pos->scalar_type() == torch::kInt32, "pos must be int32");
    s_ptr = pos->data_ptr<int>();
  }
  auto fopts = qc.options().dtype(torch::kFloat32);
  const auto at16 = [](const torch::Tensor& t) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  const bool inrow = v.data_ptr() == k.data_ptr() && vstride == Dk && Dv < Dk;
  const int tile = at16(qc) && at16(k) && at16(v) && (inrow || vstride == Dv)
                       ? attn_decode_tile(Hq / Hkv, Dk, Dv, inrow)
                       : 0;
  if (tile) {
    const long keys = s_ptr ? kScap : (long)S;
    const bool wave = Dk == Dv && attn_decode_wave(Dk, (long)B * Hkv,
                                                   window > 0 ? std::min(keys, (long)window)
                                                              : keys);
    const int nsplit = decode_slices((long)B * Hkv, keys, tile);
    torch::Tensor po, pml;
    if (nsplit > 1) {
      po = torch::empty({(long)B * Hq * nsplit * Dv}, fopts);
      pml = torch::empty({(long)B * Hq * nsplit * 2}, fopts);
    }
    launch_attn_decode_tile(
        qc.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
        nsplit > 1 ? po.data_ptr<float>() : nullptr,
        nsplit > 1 ? pml.data_ptr<float>() : nullptr, nsplit, s_ptr, B, Hq, Hkv,
        S, kScap, Dk, Dv, inrow, wave, (float)scale, (float)softcap, (int)window,
        cur_stream());
    return out;
  }
  // split-S for parallelism: target ~1024 blocks, slices of >= 512 keys
  // (>= 256 keys when B*Hkv alone leaves the chip block-starved, e.g.
  // absorbed MLA with Hkv = 1)
  long span = s_ptr ? kScap : (long)S;
  long slice = (B * Hkv <= 64) ? 256 : 512;
  int nsplit = (int)std::min<long>(
      std::min<long>(8, std::max<long>(1, 1024 / std::max(1, B * Hkv))),
      std::max<long>(1, (span + slice - 1) / slice));
  float* part_o = nullptr;
  float* part_ml = nullptr;
  torch::Tensor po, pml;
  if (nsplit > 1) {
    po = torch::empty({(long)B * Hq * nsplit * Dv}, fopts);
    pml = torch::empty({(long)B * Hq * nsplit * 2}, fopts);
    part_o = po.data_ptr<float>();
    part_ml = pml.data_ptr<float>();
  }
  launch_attn_decode(qc.data_ptr(), k.data_ptr(), v.data_ptr(),
                     out.data_ptr(), part_o, part_ml, nsplit, s_ptr, B, Hq,
                     Hkv, S, kScap, Dk, Dv, vstride, (float)scale,
                     (float)softcap, (int)window, cur_stream());
  return out;
}

// What may be fetched of the weights `ahead` [O, K] of a product of M rows behind a kernel on
// like's device: a hint, nothing where it is of another kind.
static Warm warm_of(const c10::optional<torch::Tensor>& ahead, const torch::Tensor& like,
                    long M, long K) {
  Warm warm{};
  if (ahead.has_value() && linear_few_plain(*ahead) && ahead->device() == like.device() &&
      ahead->scalar_type() == torch::kBFloat16 && ahead->dim() == 2 && ahead->size(1) == K &&
      ahead->stride(1) == 1 && ahead->stride(0) % 8 == 0 &&
      reinterpret_cast<uintptr_t>(ahead->data_ptr()) % 16 == 0 &&
      !linear_own_warm(M, ahead->size(0), K, ahead->stride(0), ahead->data_ptr(), &warm))
    warm = Warm{};
  return warm;
}

// Attention of one token per sequence from its projections on: q [B, 1, Hq, D], k and v
// [B, 1, Hkv, D] before rotations, whose row goes to the caches at pos (on the device) or
// pos0; tickets [B * Hkv] of zeros, which they are again afterwards.  [B, 1, Hq * D], or
// nothing where these are operands of the separate kernels.  ahead: weights [O, Hq * D] of
// the product behind it, which may be fetched meanwhile.
c10::optional<torch::Tensor> attn_step(
    torch::Tensor q, torch::Tensor k, torch::Tensor v, torch::Tensor cos,
    torch::Tensor sin, torch::Tensor kcache, torch::Tensor vcache,
    c10::optional<torch::Tensor> pos, int64_t pos0, torch::Tensor tickets, double scale,
    double softcap, int64_t window, bool faster, c10::optional<torch::Tensor> ahead) {
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || kcache.dim() != 4 ||
      q.size(1) != 1)
    return c10::nullopt;
  const long B = q.size(0), Hq = q.size(2), D = q.size(3), Hkv = k.size(2);
  auto whole = [](const torch::Tensor& t) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  auto on = [&](const torch::Tensor& t, at::ScalarType type) {
    return t.device() == q.device() && t.scalar_type() == type;
  };
  if (!q.is_cuda() || B < 1 || Hkv < 1 || Hq % Hkv || Hq < 1 ||
      !attn_decode_tile((int)(Hq / Hkv), (int)D, (int)D, false))
    return c10::nullopt;
  for (const auto& t : {q, k, v})
    if (!on(t, torch::kBFloat16) || t.size(0) != B || t.size(1) != 1 || t.size(3) != D ||
        t.stride(3) != 1 || t.stride(2) != D || t.stride(0) % 8 || !whole(t))
      return c10::nullopt;
  for (const auto& t : {kcache, vcache})
    if (!on(t, torch::kBFloat16) || !t.is_contiguous() || !whole(t) ||
        t.sizes() != kcache.sizes() || t.size(0) != B || t.size(1) != Hkv ||
        t.size(3) != D)
      return c10::nullopt;
  for (const auto& t : {cos, sin})
    if (!on(t, torch::kFloat32) || !t.is_contiguous() || t.numel() != D / 2 || !whole(t))
      return c10::nullopt;
  if (v.size(2) != Hkv || !on(tickets, torch::kInt32) || !tickets.is_contiguous() ||
      tickets.numel() < B * Hkv)
    return c10::nullopt;
  const long cap = kcache.size(2);
  const int* s_ptr = nullptr;
  if (pos.has_value()) {
    if (!on(*pos, torch::kInt32) || pos->numel() != 1) return c10::nullopt;
    s_ptr = pos->data_ptr<int>();
  } else {
    TORCH_CHECK(pos0 >= 0 && pos0 < cap, "no room in the cache");
  }
  // The last block of a head's merges its slices, 16 partial results a thread at once, a
  // chain of 1.3 us (heads of 256: 2.4), where the kernel of its own takes 4.5 us for any
  // number of them.  So slices are as many as two chains have, one of heads of 256, and
  // where that would be less than half of them (of heads of 256: less than all) the
  // separate kernels are faster; of heads of 256, of which a CU has one block, also for few
  // pairs with more than one slice and for more than there are CUs.  Keys are those that a
  // window leaves (1 x 56 over 8 of 128, 4279 behind a window of 1024: 12.7 us of the
  // separate kernels, 10.7 here).  Sequences x heads over heads of a size, keys:
  // us of the separate kernels, of this one with all slices, with as many as here: 1 x 8
  // over 8 of 128, 3339: 12.1, 15.9, 12.6; 1 x 32 over 8 of 128, 1970: 11.9, 12.2, 11.9;
  // 1 x 128 over 8 of 128, 757: 10.8, 13.5, 11.2; 5 x 16 over 1 of 256, 226: 11.8, 22.0;
  // 35 x 32 over 8 of 256, 89: 15.1, 21.8.  Of 1200 random sizes in captured steps 720
  // come here and take .73 of the separate kernels' time, 63 of them 3 to 16% more.  An
  // eager call takes the host 8 us and 15.8 for the separate ones, and so few keys of
  // heads of 256 (24: 7.1 us here, 5.8 there) come here, too.
  const bool wide = D == 256;
  const long pairs = B * Hkv, chains = (Hq / Hkv * D + 511) / 512;
  const int most = std::max<int>(1, (wide ? 16 : 32) / chains);
  const long held = s_ptr ? cap : pos0 + 1;
  const int slices = decode_slices(pairs, window > 0 ? std::min(held, (long)window) : held,
                                   64, wide ? 256 : 512);
  if (faster && (wide ? slices > most || (pairs < 8 && slices > 1) || pairs > 256
                      : slices > 2 * most))
    return c10::nullopt;
  const int nsplit = std::min(slices, most);
  auto out = torch::empty({B, 1, Hq * D}, q.options());
  torch::Tensor part;
  if (nsplit > 1)
    part = torch::empty({B * Hq * nsplit * (D + 2)}, q.options().dtype(torch::kFloat32));
  float* po = nsplit > 1 ? part.data_ptr<float>() : nullptr;
  const Warm warm = warm_of(ahead, q, B, Hq * D);
  launch_attn_step(q.data_ptr(), k.data_ptr(), v.data_ptr(), q.stride(0), k.stride(0),
                   v.stride(0), cos.data_ptr<float>(), sin.data_ptr<float>(),
                   kcache.data_ptr(), vcache.data_ptr(), out.data_ptr(), po,
                   po ? po + B * Hq * nsplit * D : nullptr,
                   reinterpret_cast<unsigned*>(tickets.data_ptr<int>()), nsplit, s_ptr,
                   (int)B, (int)Hq, (int)Hkv, (int)pos0 + 1, cap, (int)D, (float)scale,
                   (float)softcap, (int)window, &warm, cur_stream());
  return out;
}

// -- latent attention of one token per sequence (mla_decode.hip) -------------

// q [N, heads * (nope + rope)], latent [N, rank + rope] before norm and rotation;
// w [heads, rank, nope]; cos, sin [1, rope / 2] of the token's position; cache
// [N, 1, cap, rank + rope] gets the row at pos (on the device) or pos0.  Returns
// queries over cached rows, [N, heads, 1, rank + rope].
torch::Tensor mla_prepare(torch::Tensor q, torch::Tensor latent, torch::Tensor w,
                          torch::Tensor norm, double eps, double offset,
                          torch::Tensor cos, torch::Tensor sin,
                          torch::Tensor cache, c10::optional<torch::Tensor> pos,
                          int64_t pos0) {
  for (const auto& t : {q, latent, w, norm, cache}) check_bf16(t, "operand");
  TORCH_CHECK(q.dim() == 2 && latent.dim() == 2 && w.dim() == 3 &&
                  norm.dim() == 1 && cache.dim() == 4 && cache.size(1) == 1,
              "shapes");
  const long N = q.size(0), heads = w.size(0), rank = w.size(1), nope = w.size(2);
  const long rope = latent.size(1) - rank;
  TORCH_CHECK(N >= 1 && latent.size(0) == N && cache.size(0) == N &&
                  q.size(1) == heads * (nope + rope) && norm.size(0) == rank &&
                  cache.size(3) == rank + rope, "sizes");
  TORCH_CHECK(rank % 32 == 0 && nope % 32 == 0 && nope >= 32 && rope >= 2 &&
                  rope % 2 == 0 && (nope + rope) % 8 == 0 && (rank + rope) % 4 == 0,
              "sizes of parts");
  auto whole = [](const torch::Tensor& t) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  TORCH_CHECK(q.stride(1) == 1 && q.stride(0) % 8 == 0 && latent.stride(1) == 1 &&
                  w.is_contiguous() && norm.is_contiguous() &&
                  cache.is_contiguous() && whole(q) && whole(w) && whole(cache),
              "layout");
  TORCH_CHECK(cos.is_cuda() && sin.is_cuda() &&
                  cos.scalar_type() == torch::kFloat32 &&
                  sin.scalar_type() == torch::kFloat32 && cos.is_contiguous() &&
                  sin.is_contiguous() && cos.numel() == rope / 2 &&
                  sin.numel() == rope / 2, "one position's rotations");
  if (pos.has_value()) {
    TORCH_CHECK(pos->is_cuda() && pos->scalar_type() == torch::kInt32, "pos int32");
  } else {
    TORCH_CHECK(pos0 >= 0 && pos0 < cache.size(2), "no room in the cache");
  }
  auto out = torch::empty({N, heads, 1, rank + rope}, q.options());
  const MlaPrepareArgs a{
      (const __bf16*)q.data_ptr(), (const __bf16*)latent.data_ptr(),
      (const __bf16*)w.data_ptr(), (const __bf16*)norm.data_ptr(),
      cos.data_ptr<float>(), sin.data_ptr<float>(), (__bf16*)out.data_ptr(),
      (__bf16*)cache.data_ptr(), pos.has_value() ? pos->data_ptr<int>() : nullptr,
      q.stride(0), latent.stride(0), cache.size(2), pos0, (int)N, (int)heads,
      (int)nope, (int)rope, (int)rank, (float)eps, (float)offset};
  launch_mla_prepare(&a, cur_stream());
  return out;
}

// q from mla_prepare over the first S rows (captured: pos + 1) of the cache; w
// [heads, vdim, rank].  Returns [N, heads * vdim].
torch::Tensor mla_attend(torch::Tensor q, torch::Tensor cache, torch::Tensor w,
                         double scale, c10::optional<torch::Tensor> pos,
                         int64_t S) {
  for (const auto& t : {q, cache, w}) check_bf16(t, "operand");
  TORCH_CHECK(q.dim() == 4 && cache.dim() == 4 && w.dim() == 3, "shapes");
  const long N = q.size(0), heads = q.size(1), D = q.size(3);
  const long vdim = w.size(1), rank = w.size(2);
  const int tile = attn_decode_tile(heads, D, rank, true);
  TORCH_CHECK(tile, "no kernel for these heads");
  TORCH_CHECK(cache.size(0) == N && cache.size(1) == 1 && cache.size(3) == D &&
                  w.size(0) == heads && vdim % 16 == 0 && rank % 32 == 0, "sizes");
  for (const auto& t : {q, cache, w})
    TORCH_CHECK(t.is_contiguous() &&
                    reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0, "layout");
  const int* s_ptr = nullptr;
  if (pos.has_value()) {
    TORCH_CHECK(pos->is_cuda() && pos->scalar_type() == torch::kInt32, "pos int32");
    s_ptr = pos->data_ptr<int>();
  } else {
    TORCH_CHECK(S >= 1 && S <= cache.size(2), "rows of the cache");
  }
  const long span = s_ptr ? cache.size(2) : S;
  // A slice more is a partial result more that every block of mla_finish reads of each of
  // its up to 16 tokens, and fewer tiles one after the other: 8 sqrt(tiles / tokens) of
  // them are near the least of both, and so are all of up to five tiles (both kernels, by
  // slices: 16 sequences of 577 keys 16: 17.1 us, 10: 17.3, 8: 16.0, 4: 18.0; of 130 keys 5:
  // 13.1, 4: 13.9; 4 of 2000 56: 15.2, 32: 15.2, 16: 15.6; one of 3001 64: 12.7, 32: 13.2,
  // 16: 17.3).  Over 166 sizes 2% behind the best of 20 counts on average, 5 where there
  // are as many as CUs hold.
  const long tiles = (span + tile - 1) / tile;
  const int n = std::min(decode_slices(N, span, tile),
                         std::max(5, (int)(8.0 * std::sqrt((double)tiles / std::min(N, 16L)))));
  auto fopts = q.options().dtype(torch::kFloat32);
  auto po = torch::empty({N * heads * n, rank}, fopts);
  auto pml = torch::empty({N * heads * n, 2}, fopts);
  launch_attn_decode_tile(q.data_ptr(), cache.data_ptr(), cache.data_ptr(), nullptr,
                          po.data_ptr<float>(), pml.data_ptr<float>(), n, s_ptr,
                          (int)N, (int)heads, 1, (int)S, cache.size(2), (int)D,
                          (int)rank, true, false, (float)scale, 0.0f, 0, cur_stream());
  auto out = torch::empty({N, heads * vdim}, q.options());
  const MlaFinishArgs a{po.data_ptr<float>(), pml.data_ptr<float>(),
                        (const __bf16*)w.data_ptr(), (__bf16*)out.data_ptr(), s_ptr,
                        (int)N, (int)heads, (int)rank, (int)vdim, n, tile,
                        (int)(s_ptr ? cache.size(2) : S)};
  launch_mla_finish(&a, cur_stream());
  return out;
}

static void check_turns(const torch::Tensor& cos, const torch::Tensor& sin, long n) {
  for (const auto& t : {cos, sin})
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kFloat32 &&
                    t.is_contiguous() && t.numel() == n &&
                    reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0,
                "rotations of the prompt's positions");
}

// Rows [B, T, rank + rope] of a prompt, as projected, into the cache from row pos0 on;
// with `rows` also returned, normed, [B, T, rank].
torch::Tensor mla_rows(torch::Tensor latent, torch::Tensor norm, double eps,
                       double offset, torch::Tensor cos, torch::Tensor sin,
                       torch::Tensor cache, int64_t pos0, bool rows) {
  for (const auto& t : {latent, norm, cache}) check_bf16(t, "operand");
  TORCH_CHECK(latent.dim() == 3 && norm.dim() == 1 && cache.dim() == 4 &&
                  cache.size(1) == 1, "shapes");
  const long B = latent.size(0), T = latent.size(1), rank = norm.size(0);
  const long rope = latent.size(2) - rank;
  TORCH_CHECK(B >= 1 && T >= 1 && cache.size(0) == B &&
                  cache.size(3) == rank + rope && rank >= 8 && rank % 8 == 0 &&
                  rope >= 8 && rope % 8 == 0, "sizes");
  TORCH_CHECK(pos0 >= 0 && pos0 + T <= cache.size(2), "no room in the cache");
  auto whole = [](const torch::Tensor& t) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  TORCH_CHECK(latent.stride(2) == 1 && latent.stride(1) % 8 == 0 &&
                  (B == 1 || latent.stride(0) == T * latent.stride(1)) &&
                  norm.is_contiguous() && cache.is_contiguous() && whole(latent) &&
                  whole(norm) && whole(cache), "layout");
  check_turns(cos, sin, T * rope / 2);
  torch::Tensor out;
  if (rows) out = torch::empty({B, T, rank}, latent.options());
  const MlaRowsArgs a{
      (const __bf16*)latent.data_ptr(), (const __bf16*)norm.data_ptr(),
      cos.data_ptr<float>(), sin.data_ptr<float>(), (__bf16*)cache.data_ptr(),
      rows ? (__bf16*)out.data_ptr() : nullptr, latent.stride(1), cache.size(2),
      pos0, B * T, (int)T, (int)rank, (int)rope, (float)eps, (float)offset};
  launch_mla_rows(&a, cur_stream());
  return out;
}

// q [B, T, H, 192], unrotated; kv [B, S, H, 256]; cache [B, 1, cap, width] with S
// rows.  Returns [B, T, H * 128].
torch::Tensor mla_prompt(torch::Tensor q, torch::Tensor kv, torch::Tensor cache,
                         torch::Tensor cos, torch::Tensor sin, double scale,
                         int64_t causal_offset) {
  for (const auto& t : {q, kv, cache}) check_bf16(t, "operand");
  TORCH_CHECK(q.dim() == 4 && kv.dim() == 4 && cache.dim() == 4, "shapes");
  const long B = q.size(0), T = q.size(1), H = q.size(2), S = kv.size(1);
  TORCH_CHECK(B >= 1 && T >= 1 && H >= 1 && q.size(3) == 192 && kv.size(0) == B &&
                  kv.size(2) == H && kv.size(3) == 256 && cache.size(0) == B &&
                  cache.size(1) == 1 && cache.size(3) >= 64 &&
                  cache.size(3) % 8 == 0, "sizes");
  TORCH_CHECK(causal_offset >= 0 && causal_offset + T == S && S <= cache.size(2),
              "rows of the cache");
  for (const auto& t : {q, kv, cache})
    TORCH_CHECK(reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0, "alignment");
  TORCH_CHECK(q.stride(3) == 1 && q.stride(0) % 8 == 0 && q.stride(1) % 8 == 0 &&
                  q.stride(2) % 8 == 0 && kv.is_contiguous() &&
                  cache.is_contiguous(), "layout");
  TORCH_CHECK(H <= 65536 / 8, "row offsets of a tile in 32 bits");
  check_turns(cos, sin, T * 32);
  auto out = torch::empty({B, T, H * 128}, q.options());
  launch_mla_prompt(q.data_ptr(), kv.data_ptr(), cache.data_ptr(),
                    cos.data_ptr<float>(), sin.data_ptr<float>(), out.data_ptr(),
                    (int)B, (int)H, (int)T, (int)S, q.stride(0), q.stride(2),
                    q.stride(1), cache.size(2), (int)cache.size(3), (float)scale,
                    (int)causal_offset, cur_stream());
  return out;
}

// Attention of the long portions of a batch: q [tokens, >= H * 192], turned; k, v
// [keys, H * 128]; rows [keys, width], whose last 64 columns are the rotated key part.
// portions [n, 2] of 128 rows: request, first row.  Returns [tokens - tok_base, H * 128].
torch::Tensor latent_prompt(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                            torch::Tensor rows, torch::Tensor portions,
                            torch::Tensor cu, torch::Tensor pos0, torch::Tensor cuk,
                            int64_t n_short, int64_t tok_base, int64_t H,
                            double scale) {
  for (const auto& t : {q, k, v, rows}) {
    check_bf16(t, "operand");
    TORCH_CHECK(t.dim() == 2 && t.stride(1) == 1 &&
                    reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0, "layout");
  }
  const long keys = k.size(0);
  TORCH_CHECK(H >= 1 && H <= 8192 && q.size(1) >= H * 192 && q.stride(0) % 8 == 0 &&
                  tok_base >= 0 && tok_base < q.size(0), "queries");
  TORCH_CHECK(k.size(1) == H * 128 && v.size(0) == keys && v.size(1) == H * 128 &&
                  rows.size(0) == keys && rows.size(1) >= 64 &&
                  rows.size(1) % 8 == 0 && k.is_contiguous() && v.is_contiguous() &&
                  rows.is_contiguous(), "keys");
  auto ints = [](const torch::Tensor& t, long n) {
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kInt32 && t.is_contiguous() &&
                    t.numel() >= n, "int32 indices");
    return t.data_ptr<int>();
  };
  TORCH_CHECK(portions.dim() == 2 && portions.size(1) == 2 && portions.size(0) >= 1,
              "portions");
  auto out = torch::empty({q.size(0) - tok_base, H * 128}, q.options());
  launch_latent_prompt(q.data_ptr(), k.data_ptr(), v.data_ptr(), rows.data_ptr(),
                       out.data_ptr(), ints(portions, 2), ints(cu, n_short + 2),
                       ints(pos0, n_short + 1), ints(cuk, 2), (int)n_short,
                       (int)tok_base, (int)portions.size(0), (int)H, q.stride(0),
                       (int)rows.size(1), (float)scale, cur_stream());
  return out;
}

// q [B, Hq, T, Dk]; k/v cache views [B, Hkv, S, D] (row-contiguous)
torch::Tensor attn_prefill(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                           double scale, double softcap, int64_t window,
                           int64_t causal_offset) {
  check_bf16(q, "q");
  // rows of queries are read where they lie, in 16-byte pieces
  auto whole = [](const torch::Tensor& t) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  const bool in_place = whole(q) && q.stride(3) == 1 && q.stride(0) % 8 == 0 &&
                        q.stride(1) % 8 == 0 && q.stride(2) % 8 == 0;
  auto qc = in_place ? q : q.contiguous();
  if (!whole(qc)) qc = qc.clone();
  if (!whole(k)) k = k.clone(at::MemoryFormat::Contiguous);
  if (!whole(v)) v = v.clone(at::MemoryFormat::Contiguous);
  const int B = qc.size(0), Hq = qc.size(1), T = qc.size(2), Dk = qc.size(3);
  const int Hkv = k.size(1), S = k.size(2), Dv = v.size(3);
  TORCH_CHECK(k.stride(3) == 1 && v.stride(3) == 1, "K/V rows must be contiguous");
  TORCH_CHECK(k.stride(2) == Dk && v.stride(2) == Dv, "K/V seq stride mismatch");
  TORCH_CHECK(Hq % Hkv == 0 && Dk % 32 == 0 && Dv % 16 == 0, "shape unsupported");
  TORCH_CHECK(Dk <= 256 && Dv <= 256, "Dk<=256, Dv<=256");
  // NEVER silently skip the launch: an uninstantiated template combo
  // once fell through and returned an uninitialized output
  TORCH_CHECK(attn_prefill_supported(Dk, Dv),
              "attn_prefill: no kernel instantiation for Dk=", Dk,
              " Dv=", Dv);
  long kScap = k.stride(1) / Dk;
  long vScap = v.stride(1) / Dv;
  // heads of a token side by side, as the output projection reads them
  auto out = torch::empty({B, T, Hq, Dv}, qc.options());
  launch_attn_prefill(qc.data_ptr(), k.data_ptr(), v.data_ptr(),
                      out.data_ptr(), B, Hq, Hkv, T, S, qc.stride(0),
                      qc.stride(1), qc.stride(2), kScap, vScap, Dk, Dv,
                      (float)scale, (float)softcap, (int)window,
                      (int)causal_offset, cur_stream());
  return out.transpose(1, 2);
}

// Softmax of rows of logits [N, E]: (weights fp32, experts) of the `top` largest.
std::vector<torch::Tensor> moe_choose(torch::Tensor logits, int64_t top, double scaling,
                                      bool normalize) {
  check_bf16(logits, "logits");
  TORCH_CHECK(logits.dim() == 2 && logits.is_contiguous() && logits.size(0) >= 1 &&
                  logits.size(0) < (1L << 31) - 4 && logits.size(1) <= 64 && top >= 1 &&
                  top <= logits.size(1), "logits");
  const long N = logits.size(0);
  auto choice = torch::empty({N, top}, logits.options().dtype(torch::kInt64));
  auto weight = torch::empty({N, top}, logits.options().dtype(torch::kFloat32));
  launch_moe_choose(logits.data_ptr(), choice.data_ptr<int64_t>(),
                    weight.data_ptr<float>(), (int)N, (int)logits.size(1), (int)top,
                    normalize, (float)scaling, cur_stream());
  return {weight, choice};
}

// Routed experts of a prompt: silu(x gate^T) * (x up^T), down of that, for the pairs
// of choice [N, top] (int64).  Returns (rows [N * top, H], place of each pair).
std::vector<torch::Tensor> moe_tiles(torch::Tensor x, torch::Tensor choice,
                                     torch::Tensor gate, torch::Tensor up,
                                     torch::Tensor down, int64_t tile) {
  for (const auto& t : {x, gate, up, down}) check_bf16(t, "operand");
  TORCH_CHECK(x.dim() == 2 && choice.dim() == 2 && gate.dim() == 3 &&
                  down.dim() == 3 && gate.sizes() == up.sizes(), "shapes");
  const long N = x.size(0), H = x.size(1), top = choice.size(1);
  const long E = gate.size(0), I = gate.size(1), P = N * top;
  TORCH_CHECK(choice.size(0) == N && gate.size(2) == H && down.size(0) == E &&
                  down.size(1) == H && down.size(2) == I, "sizes");
  TORCH_CHECK(choice.is_cuda() && choice.scalar_type() == torch::kInt64 &&
                  choice.is_contiguous(), "choice: int64");
  TORCH_CHECK(H % 64 == 0 && I % 64 == 0 && H >= 128 && I >= 128 &&
                  E >= 1 && E <= MT_EXPERTS && P >= 1 && P < (1L << 30) &&
                  (tile == 128 || tile == 256), "sizes that there is no kernel for");
  TORCH_CHECK(x.stride(1) == 1 && x.stride(0) % 8 == 0 && x.stride(0) >= H &&
                  N * x.stride(0) < (1L << 31) && H * I < (1L << 31) &&
                  gate.is_contiguous() && up.is_contiguous() &&
                  down.is_contiguous(), "layout");
  for (const auto& t : {x, gate, up, down})
    TORCH_CHECK(reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0, "alignment");
  const int blocks = (int)((P + MT_BLOCK_PAIRS - 1) / MT_BLOCK_PAIRS);
  const long most = P / tile + E;  // tiles
  auto ints = torch::empty({blocks * E + 3 * most + 1 + P}, x.options().dtype(torch::kInt32));
  auto where = torch::empty({N, top}, ints.options());
  int* hist = ints.data_ptr<int>();
  int* tiles = hist + blocks * E;
  int* n_tiles = tiles + 3 * most;
  int* tokens = n_tiles + 1;
  const MoePlaceArgs place{choice.data_ptr<int64_t>(), hist, tiles, n_tiles,
                           where.data_ptr<int>(), tokens, (int)P, (int)top, (int)E,
                           blocks, (int)tile};
  launch_moe_place(&place, cur_stream());
  auto h = torch::empty({P, I}, x.options());
  auto y = torch::empty({P, H}, x.options());
  MoeTilesArgs a{(const char*)x.data_ptr(), (const char*)gate.data_ptr(),
                 (const char*)up.data_ptr(), (__bf16*)h.data_ptr(), tokens, tiles,
                 n_tiles, x.stride(0) * 2, (int)I, (int)H, 0, I * H * 2};
  launch_moe_tiles(&a, (int)tile, true, cur_stream());
  MoeTilesArgs b{(const char*)h.data_ptr(), (const char*)down.data_ptr(), nullptr,
                 (__bf16*)y.data_ptr(), nullptr, tiles, n_tiles, I * 2, (int)H,
                 (int)I, 0, I * H * 2};
  launch_moe_tiles(&b, (int)tile, false, cur_stream());
  return {y, where};
}

torch::Tensor mfma_probe(torch::Tensor A, torch::Tensor Bm) {
  check_bf16(A, "A");
  auto D = torch::empty({16, 16}, A.options().dtype(torch::kFloat32));
  launch_mfma_probe(A.contiguous().data_ptr(), Bm.contiguous().data_ptr(),
                    D.data_ptr<float>(), cur_stream());
  return D;
}

// x [M, H] bf16, wq [O, H*bits/32] uint32/int32, scales/biases [O, H/gs]
// Dense bf16 decode GEMV: y = x @ w^T on MFMA (M <= 64)
torch::Tensor dense_gemv(torch::Tensor x, torch::Tensor w) {
  check_bf16(x, "x");
  check_bf16(w, "w");
  auto xc = x.contiguous();
  const int M = xc.size(0), H = xc.size(1);
  const int O = w.size(0);
  TORCH_CHECK(w.is_contiguous(), "w must be contiguous");
  TORCH_CHECK(M <= 64 && H % 32 == 0, "dense_gemv needs M<=64, H%32==0");
  auto y = torch::empty({M, O}, xc.options());
  const int nk = bf16_gemv_nsplit(M, O, H);
  torch::Tensor yf;
  float* yfp = nullptr;
  if (nk > 1) {
    yf = torch::empty({M, O}, xc.options().dtype(torch::kFloat32));
    yfp = yf.data_ptr<float>();
  }
  launch_bf16_gemv_mfma(xc.data_ptr(), w.data_ptr(), y.data_ptr(), yfp, nk,
                        M, O, H, cur_stream());
  return y;
}

// K-segmented coalesced-A dense bf16 GEMM (gemm_kseg.hip): targets the
// K-long down_proj shapes where hipBLASLt plateaus (~3.3 TB/s)
torch::Tensor gemm_m64_kseg(torch::Tensor x, torch::Tensor w,
                            int64_t ksegs) {
  check_bf16(x, "x");
  check_bf16(w, "w");
  auto xc = x.contiguous();
  const int M = xc.size(0), K = xc.size(1);
  const int N = w.size(0);
  TORCH_CHECK(w.is_contiguous(), "w must be contiguous");
  TORCH_CHECK(M >= 1 && M <= 64 && K % 256 == 0,
              "gemm_m64_kseg needs 1<=M<=64, K%256==0");
  TORCH_CHECK(ksegs >= 1);
  auto yf = torch::empty({64, N}, xc.options().dtype(torch::kFloat32));
  auto y = torch::empty({M, N}, xc.options());
  launch_gemm_kseg(xc.data_ptr(), w.data_ptr(), yf.data_ptr<float>(),
                   y.data_ptr(), M, N, K, (int)ksegs, cur_stream());
  return y;
}

// w4a16 K-segmented GEMM: packed repacked weights (ops.repack_w4) +
// fp16 activations; bf16 out
torch::Tensor gemm_m64_kseg_w4(torch::Tensor x, torch::Tensor wq,
                               torch::Tensor sc, torch::Tensor bi,
                               int64_t gs, int64_t ksegs) {
  TORCH_CHECK(x.scalar_type() == torch::kHalf, "x must be fp16");
  auto xc = x.contiguous();
  const int M = xc.size(0), K = xc.size(1);
  const int N = wq.size(0);
  TORCH_CHECK(wq.is_contiguous() && sc.is_contiguous() && bi.is_contiguous());
  TORCH_CHECK(M >= 1 && M <= 64 && K % 256 == 0,
              "gemm_m64_kseg_w4 needs 1<=M<=64, K%256==0");
  TORCH_CHECK(gs == 32 || gs == 64 || gs == 128, "gs must be 32/64/128");
  TORCH_CHECK(wq.size(1) == K / 8, "wq must be repacked w4 [N, K/8]");
  auto yf = torch::empty({64, N}, xc.options().dtype(torch::kFloat32));
  auto y = torch::empty({M, N}, xc.options().dtype(torch::kBFloat16));
  launch_gemm_kseg_w4(xc.data_ptr(), wq.data_ptr(), sc.data_ptr(),
                      bi.data_ptr(), yf.data_ptr<float>(), y.data_ptr(), M, N,
                      K, (int)gs, (int)ksegs, cur_stream());
  return y;
}

// LDS-tiled dense bf16 GEMM, M <= 64, deep-k shapes
torch::Tensor dense_gemm64(torch::Tensor x, torch::Tensor w) {
  check_bf16(x, "x");
  check_bf16(w, "w");
  auto xc = x.contiguous();
  const int M = xc.size(0), H = xc.size(1);
  const int O = w.size(0);
  TORCH_CHECK(w.is_contiguous(), "w must be contiguous");
  TORCH_CHECK(M <= 64 && H % 8 == 0, "dense_gemm64 needs M<=64, H%8==0");
  auto y = torch::empty({M, O}, xc.options());
  const int nk = bf16_gemm_m64_nsplit(M, O, H);
  torch::Tensor yf;
  float* yfp = nullptr;
  if (nk > 1) {
    yf = torch::empty({M, O}, xc.options().dtype(torch::kFloat32));
    yfp = yf.data_ptr<float>();
  }
  launch_bf16_gemm_m64(xc.data_ptr(), w.data_ptr(), y.data_ptr(), yfp, nk, M,
                       O, H, cur_stream());
  return y;
}

torch::Tensor w4a16_gemv(torch::Tensor x, torch::Tensor wq,
                         torch::Tensor scales, torch::Tensor biases,
                         int64_t gs, int64_t bits) {
  check_bf16(x, "x");
  auto xc = x.contiguous();
  const int M = xc.size(0), H = xc.size(1);
  const int O = wq.size(0);
  auto y = torch::empty({M, O}, xc.options());
  if (M >= 8 && H % 32 == 0 && gs % 32 == 0) {
    const int nk = w4a16_mfma_nsplit(M, O, H);
    torch::Tensor yf;
    float* yfp = nullptr;
    if (nk > 1) {
      yf = torch::empty({M, O}, xc.options().dtype(torch::kFloat32));
      yfp = yf.data_ptr<float>();
    }
    launch_w4a16_mfma(xc.data_ptr(), wq.contiguous().data_ptr(),
                      scales.contiguous().data_ptr(),
                      biases.contiguous().data_ptr(), y.data_ptr(), yfp, nk,
                      M, O, H, (int)gs, (int)bits, cur_stream());
  } else {
    launch_w4a16_gemv(xc.data_ptr(), wq.contiguous().data_ptr(),
                      scales.contiguous().data_ptr(),
                      biases.contiguous().data_ptr(), y.data_ptr(), M, O, H,
                      (int)gs, (int)bits, cur_stream());
  }
  return y;
}

torch::Tensor dequant(torch::Tensor wq, torch::Tensor scales,
                      torch::Tensor biases, int64_t H, int64_t gs,
                      int64_t bits) {
  check_bf16(scales, "scales");
  check_bf16(biases, "biases");
  TORCH_CHECK(wq.is_cuda() && wq.element_size() == 4 && wq.device() == scales.device() &&
                  biases.device() == scales.device(),
              "dequant takes words of 32 bits, scales and biases on one GPU");
  const long O = wq.size(0);
  auto out = torch::empty({O, H}, scales.options());
  launch_dequant(wq.contiguous().data_ptr(), scales.contiguous().data_ptr(),
                 biases.contiguous().data_ptr(), out.data_ptr(), O, (int)H,
                 (int)gs, (int)bits, cur_stream());
  return out;
}

torch::Tensor moe_gateup_grouped(torch::Tensor x, torch::Tensor gate_w,
                                 torch::Tensor up_w, torch::Tensor sub_expert,
                                 torch::Tensor sub_off, torch::Tensor sub_cnt,
                                 torch::Tensor sorted_tok, int64_t P,
                                 int64_t max_tok) {
  check_bf16(x, "x");
  const int H = x.size(1);
  const int I = gate_w.size(1);
  const int S = sub_expert.size(0);
  TORCH_CHECK(sub_expert.scalar_type() == torch::kInt32, "sub arrays int32");
  auto h = torch::empty({P, I}, x.options());
  if (max_tok == 16 && H % 32 == 0 && I % 16 == 0) {
    launch_moe_gateup_mfma(
        x.contiguous().data_ptr(), gate_w.data_ptr(), up_w.data_ptr(),
        h.data_ptr(), sub_expert.data_ptr<int>(), sub_off.data_ptr<int>(),
        sub_cnt.data_ptr<int>(), sorted_tok.data_ptr<int>(), S, H, I,
        cur_stream());
  } else {
    TORCH_CHECK(max_tok <= 4, "scalar grouped kernel needs max_tok <= 4");
    launch_moe_gateup_grouped(
        x.contiguous().data_ptr(), gate_w.data_ptr(), up_w.data_ptr(),
        h.data_ptr(), sub_expert.data_ptr<int>(), sub_off.data_ptr<int>(),
        sub_cnt.data_ptr<int>(), sorted_tok.data_ptr<int>(), S, H, I,
        cur_stream());
  }
  return h;
}

torch::Tensor moe_down_grouped(torch::Tensor h, torch::Tensor down_w,
                               torch::Tensor sub_expert, torch::Tensor sub_off,
                               torch::Tensor sub_cnt, torch::Tensor sorted_tok,
                               torch::Tensor sorted_wt, int64_t N,
                               int64_t max_tok) {
  const int I = h.size(1);
  const int H = down_w.size(1);
  const int S = sub_expert.size(0);
  auto out = torch::zeros({N, H}, h.options().dtype(torch::kFloat32));
  if (max_tok == 16 && I % 32 == 0 && H % 16 == 0) {
    launch_moe_down_mfma(
        h.contiguous().data_ptr(), down_w.data_ptr(), out.data_ptr<float>(),
        sub_expert.data_ptr<int>(), sub_off.data_ptr<int>(),
        sub_cnt.data_ptr<int>(), sorted_tok.data_ptr<int>(),
        sorted_wt.data_ptr<float>(), S, I, H, cur_stream());
  } else {
    TORCH_CHECK(max_tok <= 4, "scalar grouped kernel needs max_tok <= 4");
    launch_moe_down_grouped(
        h.contiguous().data_ptr(), down_w.data_ptr(), out.data_ptr<float>(),
        sub_expert.data_ptr<int>(), sub_off.data_ptr<int>(),
        sub_cnt.data_ptr<int>(), sorted_tok.data_ptr<int>(),
        sorted_wt.data_ptr<float>(), S, I, H, cur_stream());
  }
  return out;
}

torch::Tensor moe_w4_mfma(torch::Tensor x, torch::Tensor wq,
                          torch::Tensor scales, torch::Tensor biases,
                          torch::Tensor sub_expert, torch::Tensor sub_off,
                          torch::Tensor sub_cnt, torch::Tensor sorted_tok,
                          int64_t P, int64_t gs, int64_t bits) {
  check_bf16(x, "x");
  const int H = x.size(1);
  const int O = wq.size(1);
  const int S = sub_expert.size(0);
  TORCH_CHECK(H % 32 == 0 && gs % 32 == 0, "H%32, gs%32 required");
  auto y = torch::empty({P, O}, x.options());
  launch_moe_w4_mfma(x.contiguous().data_ptr(), wq.data_ptr(),
                     scales.data_ptr(), biases.data_ptr(), y.data_ptr(),
                     sub_expert.data_ptr<int>(), sub_off.data_ptr<int>(),
                     sub_cnt.data_ptr<int>(), sorted_tok.data_ptr<int>(), S,
                     H, O, (int)gs, (int)bits, cur_stream());
  return y;
}

// -- routed experts of a decoding step (moe_rows.hip) -----------------------

static void check_rows(const torch::Tensor& t, const char* name, long n, long w) {
  check_bf16(t, name);
  TORCH_CHECK(t.dim() == 2 && t.size(0) == n && t.size(1) == w &&
                  t.is_contiguous() &&
                  reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0,
              name, ": contiguous rows of ", w, " at 16 bytes");
}

// x [N, H] (+ residual) -> normed rows, x + residual (or x), experts and weights
// of every token [N, top].  tickets [N]: zeros that the blocks of a token count with.
// w_in [2 S, H]: a shared feed-forward, whose units [N, S] of the normed rows come behind
// (with tickets, without a residual, up to 64 rows of 4096)
std::vector<torch::Tensor> moe_route(torch::Tensor x,
                                     c10::optional<torch::Tensor> residual,
                                     torch::Tensor norm, double eps,
                                     double offset, torch::Tensor gate,
                                     int64_t top, double scaling, bool normalize,
                                     c10::optional<torch::Tensor> tickets,
                                     c10::optional<torch::Tensor> w_in) {
  TORCH_CHECK(x.dim() == 2 && gate.dim() == 2 && norm.dim() == 1, "shapes");
  const long N = x.size(0), H = x.size(1), E = gate.size(0);
  TORCH_CHECK(N >= 1 && H % 128 == 0 && H <= 8192,
              "rows of a multiple of 128, up to 8192");
  TORCH_CHECK(E >= 1 && E <= 64 && top >= 1 && top <= E, "up to 64 experts");
  check_rows(x, "x", N, H);
  check_rows(gate, "gate", E, H);
  check_rows(norm.unsqueeze(0), "norm", 1, H);
  if (residual.has_value()) check_rows(*residual, "residual", N, H);
  auto y = torch::empty_like(x);
  auto h = residual.has_value() ? torch::empty_like(x) : x;
  auto choice = torch::empty({N, top}, x.options().dtype(torch::kInt32));
  auto weight = torch::empty({N, top}, x.options().dtype(torch::kFloat32));
  torch::Tensor logits;
  if (tickets.has_value()) {
    TORCH_CHECK(tickets->device() == x.device() && tickets->numel() == N &&
                    tickets->scalar_type() == torch::kInt32 && tickets->is_contiguous(),
                "a number per token");
    logits = torch::empty({N, 64}, weight.options());
  }
  const MoeRouteArgs a{
      (const __bf16*)x.data_ptr(),
      residual.has_value() ? (const __bf16*)residual->data_ptr() : nullptr,
      (const __bf16*)norm.data_ptr(), (const __bf16*)gate.data_ptr(),
      (__bf16*)h.data_ptr(), (__bf16*)y.data_ptr(), choice.data_ptr<int>(),
      weight.data_ptr<float>(), (int)H, (int)E, (int)top, (float)eps,
      (float)offset, (float)scaling, normalize,
      tickets.has_value() ? logits.data_ptr<float>() : nullptr,
      tickets.has_value() ? reinterpret_cast<unsigned*>(tickets->data_ptr<int>()) : nullptr};
  if (!w_in.has_value()) {
    launch_moe_route(&a, (int)N, cur_stream());
    return {y, h, choice, weight};
  }
  TORCH_CHECK(tickets.has_value() && !residual.has_value() && N <= 64 && H <= 4096 &&
                  w_in->device() == x.device(),
              "rows that a shared feed-forward goes with");
  const long S = w_in->size(0) / 2;
  TORCH_CHECK(S >= 1 && S < 1L << 24, "units");
  check_rows(*w_in, "w_in", 2 * S, H);
  auto units = torch::empty({N, S}, x.options());
  launch_moe_begin(&a, (int)N, w_in->data_ptr(), units.data_ptr(), (int)S, cur_stream());
  return {y, h, choice, weight, units};
}

// Packed words [E, O, K * bits / 32] with scales and offsets [E, O, K / gs] in the
// order of moe_rows.hip: [E, O / 16, K / 128, words of a tile]
torch::Tensor moe_pack(torch::Tensor w, torch::Tensor scales,
                       torch::Tensor offsets, int64_t bits, int64_t gs) {
  TORCH_CHECK(bits == 4 || bits == 8, "4 or 8 bits");
  TORCH_CHECK(gs == 32 || gs == 64 || gs == 128, "group size");
  TORCH_CHECK(w.is_cuda() && w.dim() == 3 && w.element_size() == 4 &&
                  w.is_contiguous() &&
                  reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
              "packed words, contiguous, at 16 bytes");
  const long E = w.size(0), O = w.size(1), K = w.size(2) * 32 / bits;
  TORCH_CHECK(K % 128 == 0 && O % 16 == 0, "whole tiles");
  for (const auto& t : {scales, offsets}) {
    check_bf16(t, "scales and offsets");
    TORCH_CHECK(t.dim() == 3 && t.is_contiguous() && t.size(0) == E &&
                    t.size(1) == O && t.size(2) == K / gs, "one per group");
  }
  auto out = torch::empty({E, O / 16, K / 128, moe_pack_words(bits, gs)},
                          w.options().dtype(torch::kInt32));
  if (out.numel())
    launch_moe_pack(w.data_ptr(), scales.data_ptr(), offsets.data_ptr(),
                    out.data_ptr(), (int)(E * O), (int)K, (int)bits, (int)gs,
                    cur_stream());
  return out;
}

// One stack of experts' matrices: from moe_pack, or bf16 [E, O, K]
struct ExpertStack {
  const void* w;
  long E, O, K;
};

static ExpertStack expert_stack(const torch::Tensor& t, int bits, int gs) {
  TORCH_CHECK(t.is_cuda() && t.is_contiguous() &&
                  reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0,
              "stacks are contiguous, at 16 bytes");
  ExpertStack s{t.data_ptr(), t.size(0), 0, 0};
  if (bits == 16) {
    check_bf16(t, "weights");
    TORCH_CHECK(t.dim() == 3, "a stack");
    s.O = t.size(1);
    s.K = t.size(2);
  } else {
    TORCH_CHECK(t.dim() == 4 && t.scalar_type() == torch::kInt32 &&
                    t.size(3) == moe_pack_words(bits, gs), "a packed stack");
    s.O = t.size(1) * 16;
    s.K = t.size(2) * 128;
  }
  TORCH_CHECK(s.K % 128 == 0 && s.O % 16 == 0 && s.K >= 128 && s.O >= 16 &&
                  s.K <= moe_rows_longest(bits), "sizes of an expert");
  return s;
}

// Every pair's expert output, weighted, fp32 [N * top, H]; bits 16: bf16 stacks.
// shared_in [2 S, H], shared_out [H, S]: a feed-forward that all tokens (up to 8) pass,
// whose bf16 rows [N, H] come behind (no rows without).
std::vector<torch::Tensor> moe_rows(torch::Tensor x, torch::Tensor choice,
                                    torch::Tensor weight, torch::Tensor gate,
                                    torch::Tensor up, torch::Tensor down, int64_t bits,
                                    int64_t gs, c10::optional<torch::Tensor> shared_in,
                                    c10::optional<torch::Tensor> shared_out) {
  TORCH_CHECK(bits == 4 || bits == 8 || bits == 16, "4, 8 or 16 bits");
  TORCH_CHECK(bits == 16 || gs == 32 || gs == 64 || gs == 128, "group size");
  const auto g = expert_stack(gate, bits, gs), u = expert_stack(up, bits, gs),
             d = expert_stack(down, bits, gs);
  TORCH_CHECK(g.E == u.E && g.O == u.O && g.K == u.K && d.E == g.E &&
                  d.O == g.K && d.K == g.O && g.E <= 64, "stacks of one shape");
  TORCH_CHECK(choice.dim() == 2 && choice.is_contiguous() &&
                  choice.scalar_type() == torch::kInt32 && choice.is_cuda() &&
                  weight.sizes() == choice.sizes() && weight.is_contiguous() &&
                  weight.scalar_type() == torch::kFloat32 && weight.is_cuda(),
              "choice int32, weight fp32 [N, top]");
  const long N = choice.size(0), P = choice.numel();
  TORCH_CHECK(P >= 1 && P <= MR_PAIRS, "up to ", MR_PAIRS, " pairs");
  check_rows(x, "x", N, g.K);
  TORCH_CHECK(shared_in.has_value() == shared_out.has_value(), "both or none");
  const long S = shared_in.has_value() ? shared_out->size(-1) : 0;
  if (shared_in.has_value()) {
    TORCH_CHECK(N <= 8 && S >= 64 && S % 64 == 0 && std::max(S, g.K) <= 16 * 256,
                "sizes of the shared feed-forward");
    check_rows(*shared_in, "shared_in", 2 * S, g.K);
    check_rows(*shared_out, "shared_out", g.K, S);
  }
  auto h = torch::empty({P, g.O}, x.options().dtype(bits == 16 ? torch::kBFloat16
                                                                : torch::kHalf));
  auto y = torch::empty({P, d.O}, x.options().dtype(torch::kFloat32));
  auto hs = torch::empty({N, S}, x.options());
  auto ys = torch::empty({S ? N : 0, d.O}, x.options());
  MoeRowsArgs a{x.data_ptr(), g.w, u.w, h.data_ptr(),
                choice.data_ptr<int>(), weight.data_ptr<float>(), (int)P,
                (int)choice.size(1), (int)g.E, (int)g.O, (int)g.K};
  if (S) {
    a.dx = (const __bf16*)x.data_ptr();
    a.dw = (const __bf16*)shared_in->data_ptr();
    a.dy = (__bf16*)hs.data_ptr();
    a.dense = (int)S / 16;
    a.N = (int)N;
    a.DO = (int)S;
    a.DK = (int)g.K;
  }
  launch_moe_rows(&a, (int)bits, (int)gs, true, cur_stream());
  MoeRowsArgs b{h.data_ptr(), d.w, nullptr, y.data_ptr(), choice.data_ptr<int>(),
                weight.data_ptr<float>(), (int)P, (int)choice.size(1), (int)d.E,
                (int)d.O, (int)d.K};
  if (S) {
    b.dx = (const __bf16*)hs.data_ptr();
    b.dw = (const __bf16*)shared_out->data_ptr();
    b.dy = (__bf16*)ys.data_ptr();
    b.dense = (int)d.O / 16;
    b.N = (int)N;
    b.DO = (int)d.O;
    b.DK = (int)S;
  }
  launch_moe_rows(&b, (int)bits, (int)gs, false, cur_stream());
  return {y, ys};
}

// units [N, S] w_out [H, S]^T, a token's pairs [N * top, H] and the rows h, added up in 32 bits
torch::Tensor moe_finish(torch::Tensor units, torch::Tensor w_out, torch::Tensor rows,
                         torch::Tensor h) {
  TORCH_CHECK(units.dim() == 2 && w_out.dim() == 2 && rows.dim() == 2, "shapes");
  const long N = units.size(0), S = units.size(1), H = w_out.size(0);
  TORCH_CHECK(N >= 1 && N <= 64 && S >= 32 && S % 32 == 0 && S <= 65536 && H >= 16 &&
                  H % 16 == 0 && H < 1L << 24, "sizes of the shared feed-forward");
  check_rows(units, "units", N, S);
  check_rows(w_out, "w_out", H, S);
  check_rows(h, "h", N, H);
  TORCH_CHECK(w_out.device() == units.device() && h.device() == units.device(), "one device");
  TORCH_CHECK(rows.is_cuda() && rows.device() == units.device() &&
                  rows.scalar_type() == torch::kFloat32 && rows.is_contiguous() &&
                  rows.size(1) == H && rows.size(0) >= N && rows.size(0) % N == 0, "rows");
  auto out = torch::empty({N, H}, units.options());
  launch_moe_finish(units.data_ptr(), w_out.data_ptr(), rows.data_ptr<float>(), h.data_ptr(),
                    out.data_ptr(), (int)N, (int)H, (int)S, (int)(rows.size(0) / N),
                    cur_stream());
  return out;
}

// A token's pairs, and the rows h and shared where given, added up in 32 bits
torch::Tensor moe_combine(torch::Tensor rows, c10::optional<torch::Tensor> h,
                          c10::optional<torch::Tensor> shared, int64_t N) {
  TORCH_CHECK(rows.is_cuda() && rows.scalar_type() == torch::kFloat32 &&
                  rows.dim() == 2 && rows.is_contiguous() && N >= 1 &&
                  rows.size(0) % N == 0 && rows.size(1) % 4 == 0, "rows");
  const long H = rows.size(1);
  if (h.has_value()) check_rows(*h, "h", N, H);
  if (shared.has_value()) check_rows(*shared, "shared", N, H);
  auto out = torch::empty({N, H}, rows.options().dtype(torch::kBFloat16));
  launch_moe_combine(rows.data_ptr<float>(), h.has_value() ? h->data_ptr() : nullptr,
                     shared.has_value() ? shared->data_ptr() : nullptr,
                     out.data_ptr(), (int)N, (int)H, (int)(rows.size(0) / N),
                     cur_stream());
  return out;
}

// Fused fp16-dequant gate+up+SiLU over repacked quant words.
// x [N, H] fp16; gq/uq [E, I, H*bits/32] repacked; scales/biases bf16.
torch::Tensor moe_w4f16_gateup(torch::Tensor x, torch::Tensor gq,
                               torch::Tensor uq, torch::Tensor gsc,
                               torch::Tensor gbi, torch::Tensor usc,
                               torch::Tensor ubi, torch::Tensor sub_expert,
                               torch::Tensor sub_off, torch::Tensor sub_cnt,
                               torch::Tensor sorted_tok, int64_t P,
                               int64_t gs, int64_t bits) {
  TORCH_CHECK(x.scalar_type() == torch::kHalf, "x must be fp16");
  const int H = x.size(1);
  const int I = gq.size(1);
  const int S = sub_expert.size(0);
  TORCH_CHECK(H % 32 == 0, "H%32 required");
  TORCH_CHECK(gs == 32 || gs == 64 || gs == 128, "gs must be 32/64/128");
  auto h = torch::empty({P, I}, x.options());
  launch_moe_w4f16_gateup(
      x.contiguous().data_ptr(), gq.data_ptr(), uq.data_ptr(), gsc.data_ptr(),
      gbi.data_ptr(), usc.data_ptr(), ubi.data_ptr(), h.data_ptr(),
      sub_expert.data_ptr<int>(), sub_off.data_ptr<int>(),
      sub_cnt.data_ptr<int>(), sorted_tok.data_ptr<int>(), S, H, I, (int)gs,
      (int)bits, cur_stream());
  return h;
}

torch::Tensor moe_w4f16_down(torch::Tensor hh, torch::Tensor dq,
                             torch::Tensor dsc, torch::Tensor dbi,
                             torch::Tensor sub_expert, torch::Tensor sub_off,
                             torch::Tensor sub_cnt, torch::Tensor sorted_tok,
                             torch::Tensor sorted_wt, int64_t N, int64_t gs,
                             int64_t bits) {
  TORCH_CHECK(hh.scalar_type() == torch::kHalf, "h must be fp16");
  const int I = hh.size(1);
  const int H = dq.size(1);
  const int S = sub_expert.size(0);
  TORCH_CHECK(I % 32 == 0, "I%32 required");
  TORCH_CHECK(gs == 32 || gs == 64 || gs == 128, "gs must be 32/64/128");
  auto out = torch::zeros({N, H}, hh.options().dtype(torch::kFloat32));
  launch_moe_w4f16_down(
      hh.contiguous().data_ptr(), dq.data_ptr(), dsc.data_ptr(),
      dbi.data_ptr(), out.data_ptr<float>(), sub_expert.data_ptr<int>(),
      sub_off.data_ptr<int>(), sub_cnt.data_ptr<int>(),
      sorted_tok.data_ptr<int>(), sorted_wt.data_ptr<float>(), S, I, H,
      (int)gs, (int)bits, cur_stream());
  return out;
}

// Dense fp16-dequant w4/w8 GEMV: x [M, H] fp16, wq REPACKED
// (ops.repack_w4), scales/biases bf16.  Returns bf16 [M, O].
torch::Tensor w4f16_gemv(torch::Tensor x, torch::Tensor wq,
                         torch::Tensor scales, torch::Tensor biases,
                         int64_t gs, int64_t bits) {
  TORCH_CHECK(x.scalar_type() == torch::kHalf, "x must be fp16");
  auto xc = x.contiguous();
  const int M = xc.size(0), H = xc.size(1);
  const int O = wq.size(0);
  TORCH_CHECK(M <= 64 && H % 32 == 0, "w4f16_gemv needs M<=64, H%32==0");
  TORCH_CHECK(gs == 32 || gs == 64 || gs == 128, "gs must be 32/64/128");
  auto y = torch::empty({M, O},
                        xc.options().dtype(torch::kBFloat16));
  const int nk = w4f16_gemv_nsplit(M, O, H);
  torch::Tensor yf;
  float* yfp = nullptr;
  if (nk > 1) {
    yf = torch::empty({M, O}, xc.options().dtype(torch::kFloat32));
    yfp = yf.data_ptr<float>();
  }
  launch_w4f16_gemv(xc.data_ptr(), wq.contiguous().data_ptr(),
                    scales.contiguous().data_ptr(),
                    biases.contiguous().data_ptr(), y.data_ptr(), yfp, nk, M,
                    O, H, (int)gs, (int)bits, cur_stream());
  return y;
}

std::vector<torch::Tensor> moe_gate_subranges(torch::Tensor logits, int64_t K,
                                              int64_t s_upper, int64_t max_tok,
                                              double routed_scaling,
                                              bool norm_topk) {
  check_bf16(logits, "logits");
  auto lc = logits.contiguous();
  const int N = lc.size(0), E = lc.size(1);
  TORCH_CHECK(N <= 128 && E <= 64 && K <= 8,
              "fused gate limits: N<=128, E<=64, K<=8");
  const long P = (long)N * K;
  auto opts = torch::TensorOptions().dtype(torch::kInt32).device(lc.device());
  auto sorted_tok = torch::empty({P}, opts);
  auto sorted_wt = torch::empty({P}, opts.dtype(torch::kFloat32));
  auto sub_expert = torch::empty({s_upper}, opts);
  auto sub_off = torch::empty({s_upper}, opts);
  auto sub_cnt = torch::empty({s_upper}, opts);
  launch_moe_gate_subranges(lc.data_ptr(), sorted_tok.data_ptr<int>(),
                            sorted_wt.data_ptr<float>(),
                            sub_expert.data_ptr<int>(), sub_off.data_ptr<int>(),
                            sub_cnt.data_ptr<int>(), N, E, (int)K,
                            (int)s_upper, (int)max_tok, (float)routed_scaling,
                            norm_topk ? 1 : 0, cur_stream());
  return {sub_expert, sub_off, sub_cnt, sorted_tok, sorted_wt};
}

}  // namespace

// A layer's attention of few tokens that are no single ones, in one call: the products of
// x's rows, as the norm makes them, with w_qkv (queries, keys, values of all heads), their
// rotations, keys and values to the caches from place `at` on, attention, and w_o's product,
// plus the residual.  Nothing, and nothing written, where one of these does not run here.
// (Launched one by one from Python, six kernels of a layer took the host 70 us, four in this
// call and a feed-forward 38; three are left.)
c10::optional<torch::Tensor> attend_few_try(
    torch::Tensor x, torch::Tensor w_qkv, c10::optional<torch::Tensor> b_qkv,
    torch::Tensor norm, double eps, double offset, torch::Tensor cos, torch::Tensor sin,
    torch::Tensor kcache, torch::Tensor vcache, int64_t at, torch::Tensor w_o,
    c10::optional<torch::Tensor> b_o, c10::optional<torch::Tensor> residual, int64_t heads,
    double scale, double softcap, int64_t window) {
  if (x.dim() != 3 || kcache.dim() != 4 || !linear_few_input(x) ||
      !linear_few_weight(w_qkv, x) || !linear_few_weight(w_o, x) || w_qkv.size(1) < 1 ||
      x.size(2) != w_qkv.size(1) ||
      !linear_few_more(x.numel() / x.size(2), w_qkv.size(0), x.size(2), 0))
    return {};
  const long B = x.size(0), T = x.size(1), M = B * T, Hkv = kcache.size(1),
             cap = kcache.size(2), D = kcache.size(3), wide = (heads + 2 * Hkv) * D;
  if (heads < 1 || Hkv < 1 || heads % Hkv || D < 32 || D % 32 || D > 256 ||
      !attn_prefill_supported((int)D, (int)D) || w_qkv.size(0) != wide ||
      w_o.size(1) != heads * D || !linear_few_more(M, w_o.size(0), heads * D, 0) ||
      !linear_turned_takes(M, heads + 2 * Hkv, D, x.size(2)) ||
      !linear_few_along(x, wide, wide, b_qkv, {}, norm) ||
      !linear_few_along(x, w_o.size(0), w_o.size(0), b_o, residual, {}) || at < 0 ||
      at + T > cap)
    return {};
  for (const auto& t : {kcache, vcache})
    if (t.device() != x.device() || t.scalar_type() != torch::kBFloat16 || t.dim() != 4 ||
        t.size(0) != B || t.size(1) != Hkv || t.size(2) != cap || t.size(3) != D ||
        !t.is_contiguous() || !linear_few_whole(t) || !linear_few_plain(t))
      return {};
  for (const auto& t : {cos, sin})
    if (t.device() != x.device() || t.scalar_type() != torch::kFloat32 ||
        !t.is_contiguous() || t.numel() != T * D / 2 || !linear_few_plain(t))
      return {};
  c10::OptionalDeviceGuard guard;  // and the device's current stream
  if (x.get_device() != c10::hip::current_device()) guard.reset_device(x.device());
  const auto q = torch::empty({M, heads * D}, x.options());
  const auto rows = linear_few_rows(x);
  const TurnedArgs t{cos.data_ptr<float>(), sin.data_ptr<float>(), (__bf16*)kcache.data_ptr(),
                     (__bf16*)vcache.data_ptr(), cap, at, (int)T, (int)heads, (int)Hkv};
  launch_linear_turned(rows.data_ptr(), w_qkv.data_ptr(),
                       b_qkv.has_value() ? b_qkv->data_ptr() : nullptr, norm.data_ptr(),
                       q.data_ptr(), (int)M, (int)w_qkv.size(1), (int)D, rows.stride(0),
                       w_qkv.stride(0), (float)eps, (float)offset, &t, cur_stream());
  const auto o = torch::empty({M, heads * D}, x.options());
  launch_attn_prefill(q.data_ptr(), kcache.data_ptr(), vcache.data_ptr(), o.data_ptr(), (int)B,
                      (int)heads, (int)Hkv, (int)T, (int)(at + T), T * heads * D, D, heads * D,
                      cap, cap, (int)D, (int)D, (float)scale, (float)softcap, (int)window,
                      (int)at, cur_stream());
  if (residual.has_value()) residual = residual->reshape({M, -1});
  return linear_few_shaped(linear_few_run(o, w_o, b_o, residual, {}, 0.0, 0.0, 0, {}, {}), x);
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rms_norm", &rms_norm, "fused RMSNorm (gfx950)");
  m.def("norm_add", &norm_add);
  m.def("attn_step", &attn_step);
  m.def("attend_few_try", &attend_few_try);
  m.def("linear_own_many", [](int64_t M, int64_t O, int64_t K, int64_t act) {
    return (bool)linear_own_many(M, O, K, (int)act);
  });
  m.def("step_begin", &step_begin);
  m.def("step_end", &step_end);
  m.def("rope_qkv", &rope_qkv, py::arg("q"), py::arg("k"), py::arg("v"),
        py::arg("cos"), py::arg("sin"), py::arg("kcache"), py::arg("vcache"),
        py::arg("pos") = py::none(), py::arg("pos0") = 0);
  m.def("rms_norm_residual", &rms_norm_residual);
  m.def("glu", &glu);
  m.def("softcap", &softcap_op);
  m.def("apply_rope", &apply_rope);
  m.def("rope_append_kv", &rope_append_kv, pybind11::arg("k"),
        pybind11::arg("v"), pybind11::arg("cos"), pybind11::arg("sin"),
        pybind11::arg("kcache"), pybind11::arg("vcache"),
        pybind11::arg("pos") = pybind11::none(), pybind11::arg("pos0") = 0,
        pybind11::arg("interleaved") = false);
  m.def("mla_append_kv", &mla_append_kv,
        pybind11::arg("kvh"), pybind11::arg("kpe"), pybind11::arg("kcache"),
        pybind11::arg("vcache"), pybind11::arg("pos") = pybind11::none(),
        pybind11::arg("pos0") = 0);
  m.def("attn_decode", &attn_decode, pybind11::arg("q"), pybind11::arg("k"),
        pybind11::arg("v"), pybind11::arg("scale"), pybind11::arg("softcap"),
        pybind11::arg("window"), pybind11::arg("pos") = pybind11::none());
  m.def("attn_decode_shape_ok", [](int64_t g, int64_t dv) {
    return attn_decode_supported_shape((int)g, (int)dv);
  });
  m.def("attn_prefill", &attn_prefill);
  m.def("attn_prefill_shape_ok", [](int64_t dk, int64_t dv) {
    return attn_prefill_supported((int)dk, (int)dv);
  });
  m.def("linear_few_try", &linear_few_try, py::arg("x"), py::arg("w"), py::arg("bias"),
        py::arg("residual"), py::arg("norm"), py::arg("eps"), py::arg("offset"),
        py::arg("act"), py::arg("clear") = py::none());
  m.def("linear_clamped_try", &linear_clamped_try);
  m.def("feed_few_try", &feed_few_try);
  m.def("mla_rows", &mla_rows);
  m.def("mla_prompt", &mla_prompt);
  m.def("latent_prompt", &latent_prompt);
  m.def("mla_prepare", &mla_prepare);
  m.def("mla_attend", &mla_attend);
  m.def("attn_decode_tile", [](int64_t g, int64_t dk, int64_t dv, bool inrow) {
    return attn_decode_tile((int)g, (int)dk, (int)dv, inrow);
  });
  m.def("moe_route", &moe_route, py::arg("x"), py::arg("residual"), py::arg("norm"),
        py::arg("eps"), py::arg("offset"), py::arg("gate"), py::arg("top"),
        py::arg("scaling"), py::arg("normalize"), py::arg("tickets") = py::none(),
        py::arg("w_in") = py::none());
  m.def("moe_pack", &moe_pack);
  m.def("moe_rows", &moe_rows);
  m.def("moe_rows_longest", [](int64_t bits) { return moe_rows_longest((int)bits); });
  m.def("moe_combine", &moe_combine);
  m.def("moe_finish", &moe_finish);
  m.def("moe_tiles", &moe_tiles);
  m.def("linear_tiles", &linear_tiles);
  m.def("linear_tiles_plan", &linear_tiles_planned);
  m.def("mfma_probe", &mfma_probe);
  m.def("w4a16_gemv", &w4a16_gemv);
  m.def("w4f16_gemv", &w4f16_gemv);
  m.def("dense_gemv", &dense_gemv);
  m.def("dense_gemm64", &dense_gemm64);
  m.def("gemm_m64_kseg", &gemm_m64_kseg);
  m.def("gemm_m64_kseg_w4", &gemm_m64_kseg_w4);
  m.def("dequant", &dequant);
  m.def("moe_gateup_grouped", &moe_gateup_grouped);
  m.def("moe_down_grouped", &moe_down_grouped);
  m.def("moe_w4_mfma", &moe_w4_mfma);
  m.def("moe_w4f16_gateup", &moe_w4f16_gateup);
  m.def("moe_w4f16_down", &moe_w4f16_down);
  m.def("moe_gate_subranges", &moe_gate_subranges);
  m.def("moe_scatter_rows",
        [](torch::Tensor src, torch::Tensor dst, torch::Tensor src_idx,
           torch::Tensor dst_idx) {
          check_bf16(src, "src");
          const int P = src_idx.size(0), H = src.size(-1);
          TORCH_CHECK(H % 4 == 0 && dst.size(-1) == H, "row shape");
          TORCH_CHECK(src_idx.scalar_type() == torch::kInt32 &&
                          dst_idx.scalar_type() == torch::kInt32,
                      "indices int32");
          launch_moe_scatter_rows(src.contiguous().data_ptr(), dst.data_ptr(),
                                  src_idx.data_ptr<int>(),
                                  dst_idx.data_ptr<int>(), P, H,
                                  cur_stream());
        });
  m.def("moe_gather_reduce",
        [](torch::Tensor d, torch::Tensor pos, torch::Tensor wts, int64_t N,
           c10::optional<torch::Tensor> plus, c10::optional<torch::Tensor> plus2) {
          check_bf16(d, "d");
          const int K = pos.size(1), H = d.size(-1);
          TORCH_CHECK(pos.scalar_type() == torch::kInt32, "pos int32");
          TORCH_CHECK(wts.scalar_type() == torch::kFloat32, "wts fp32");
          auto rows = [&](const c10::optional<torch::Tensor>& t) -> const void* {
            if (!t.has_value()) return nullptr;
            check_bf16(*t, "rows to add");
            TORCH_CHECK(t->is_contiguous() && t->numel() == N * H &&
                            reinterpret_cast<uintptr_t>(t->data_ptr()) % 8 == 0,
                        "rows to add");
            return t->data_ptr();
          };
          auto out = torch::empty({N, H}, d.options());
          launch_moe_gather_reduce(d.contiguous().data_ptr(),
                                   pos.contiguous().data_ptr<int>(),
                                   wts.contiguous().data_ptr<float>(), rows(plus),
                                   rows(plus2), out.data_ptr(), (int)N, K, H,
                                   cur_stream());
          return out;
        }, py::arg("d"), py::arg("pos"), py::arg("wts"), py::arg("N"),
        py::arg("plus") = py::none(), py::arg("plus2") = py::none());
  m.def("moe_choose", &moe_choose);
}
