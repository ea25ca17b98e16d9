// y = x W^T for up to 64 rows, with what goes with it (linear_few.hip, linear_own.hip), and
// for more where linear_own.hip or linear_tiles.hip is the better one; part of both extensions.
#pragma once

#include <torch/extension.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <cstdlib>
#include <cstring>

#include "linear_tiles.h"

extern "C" void launch_linear_few(const void*, const void*, const void*,
                                  const void*, const void*, void*, int, int, int,
                                  long, long, long, long, float, float, int,
                                  unsigned*, float*, unsigned*, int, hipStream_t);
extern "C" long linear_few_room(int, int, int, int*);
extern "C" int linear_own_many(long, long, long, int);

// Room for a product whose contraction blocks share; whatever runs before it clears the
// numbers.
struct LinearFewRoom {
  torch::Tensor held;
  unsigned* numbers = nullptr;
  float* sums = nullptr;
  int n = 0;

  LinearFewRoom() = default;
  LinearFewRoom(int M, int O, int K, const torch::Tensor& like) {
    const long floats = linear_few_room(M, O, K, &n);
    if (!n) return;
    const long at = (n + 63) / 64 * 64;
    held = torch::empty({at + floats}, like.options().dtype(torch::kFloat32));
    numbers = reinterpret_cast<unsigned*>(held.data_ptr<float>());
    sums = held.data_ptr<float>() + at;
  }
};

// x [M, K], w [O, K] (act: [2 O, K]); bias per row of w, residual [M, O], norm
// weights [K] for the rows of x; act 0: none, 1: silu, 2: gelu_tanh, 3: clamped, by eps and
// offset (LF_CLAMPED), without a norm, its bias the gate's and `up` the up projection's, of the
// first columns each (the others have none).  room: for a shared contraction; clear: the numbers
// of another one's that runs behind this.
static torch::Tensor linear_few_run(const torch::Tensor& x, const torch::Tensor& w,
                                    const c10::optional<torch::Tensor>& bias,
                                    const c10::optional<torch::Tensor>& residual,
                                    const c10::optional<torch::Tensor>& norm, double eps,
                                    double offset, int64_t act, const LinearFewRoom& room,
                                    const LinearFewRoom& clear,
                                   const c10::optional<torch::Tensor>& up = {}) {
  auto bf16 = [&](const torch::Tensor& t) {
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kBFloat16 &&
                    t.device() == x.device(),
                "linear_few takes bf16 tensors on one GPU");
  };
  auto whole = [](const torch::Tensor& t) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  bf16(x);
  bf16(w);
  TORCH_CHECK(act >= 0 && act <= (norm || room.n ? 2 : 3), "unknown unit");
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1), "shapes");
  const int M = x.size(0), K = x.size(1), O = w.size(0) / (act ? 2 : 1);
  TORCH_CHECK(M >= 1 && K >= 32 && K % 32 == 0 && O >= 1 &&
                  (M <= 64 || (!room.n && linear_own_many(M, O, K, (int)act))),
              "1 to 64 rows of a multiple of 32, or more that there is a kernel for");
  TORCH_CHECK(!act || w.size(0) % 2 == 0, "a gated unit has two halves");
  for (const auto& t : {x, w})
    TORCH_CHECK(t.stride(1) == 1 && t.stride(0) % 8 == 0 && whole(t),
                "rows of x and w begin at multiples of 16 bytes");
  auto vec = [&](const c10::optional<torch::Tensor>& t, long n) -> const void* {
    if (!t.has_value()) return nullptr;
    bf16(*t);
    TORCH_CHECK(t->is_contiguous() && t->numel() == n, "size of a vector");
    return t->data_ptr();
  };
  const long biased = act == 3 && bias ? bias->numel() : w.size(0);
  TORCH_CHECK(act != 3 || (bias.has_value() == up.has_value() && !residual && !clear.n &&
                           (!bias || (biased >= 1 && biased <= O))),
              "both halves of a clamped unit have a bias, or none");
  const void* b = vec(bias, biased);
  const void* n = vec(norm, K);
  TORCH_CHECK(!n || (whole(*norm) && K <= 32768),
              "norm weights begin at a multiple of 16 bytes, up to 32768 of them");
  const void* r = nullptr;
  long ldr = 0;
  if (residual.has_value()) {
    bf16(*residual);
    TORCH_CHECK(residual->dim() == 2 && residual->size(0) == M &&
                    residual->size(1) == O && residual->stride(1) == 1,
                "shape of the residual");
    r = residual->data_ptr();
    ldr = residual->stride(0);
  }
  if (act == 3) r = vec(up, biased);  // (LF_CLAMPED)
  c10::OptionalDeviceGuard guard;  // and the device's current stream
  if (x.get_device() != c10::hip::current_device()) guard.reset_device(x.device());
  auto y = torch::empty({M, O}, x.options());
  launch_linear_few(x.data_ptr(), w.data_ptr(), b, r, n, y.data_ptr(), M, O, K,
                    x.stride(0), w.stride(0), ldr, O, (float)eps, (float)offset,
                    (int)act, room.numbers, room.sums, clear.numbers,
                    act == 3 ? (int)biased : clear.n,
                    c10::hip::getCurrentHIPStream().stream());
  return y;
}

// An ordinary tensor that nothing differentiates, maps or traces.
static bool linear_few_plain(const torch::Tensor& t) {
  static const c10::DispatchKeySet odd({
      c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
      c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
      c10::DispatchKey::Batched, c10::DispatchKey::Conjugate,
      c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
  return !t.key_set().has_any(odd) &&
         !(t.requires_grad() && at::GradMode::is_enabled());
}

// Whether torch.jit.trace or a dispatch mode records this thread's operators.
static bool linear_few_recorded() {
  static const c10::DispatchKeySet recorders(
      {c10::DispatchKey::Python, c10::DispatchKey::Tracer});
  return c10::impl::tls_local_dispatch_key_set().included_.has_any(recorders);
}

// Whether the environment asks for other kernels, or for torch's own.
static bool linear_few_other(long K) {
  auto is = [](const char* name, const char* value) {
    const char* v = std::getenv(name);
    return v && *v && (!value || !std::strcmp(v, value));
  };
  return is("MLXS_AMD_FORCE_TORCH", "1") || is("MLXS_AMD_DENSE_GEMV", nullptr) ||
         (K >= 16384 && is("MLXS_AMD_GEMM64", nullptr));
}

static bool linear_few_whole(const torch::Tensor& t) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

// Whether x's rows can be read here: bf16, beginning at whole 16-byte vectors.
static bool linear_few_input(const torch::Tensor& x) {
  if (!x.is_cuda() || x.scalar_type() != torch::kBFloat16 || x.dim() < 1 ||
      !linear_few_plain(x) || linear_few_recorded())
    return false;
  if (at::autocast::is_autocast_enabled(at::kCUDA) &&
      at::autocast::get_autocast_dtype(at::kCUDA) != at::kBFloat16)
    return false;  // a product of another type
  for (long d = 0; d + 1 < x.dim(); ++d)
    if (x.stride(d) % 8) return false;
  return x.stride(-1) == 1 && linear_few_whole(x);
}

static bool linear_few_weight(const torch::Tensor& w, const torch::Tensor& x) {
  return w.device() == x.device() && w.scalar_type() == torch::kBFloat16 &&
         w.dim() == 2 && linear_few_plain(w) && w.stride(1) == 1 &&
         w.stride(0) % 8 == 0 && linear_few_whole(w);
}

// Whether a product of this size runs here.  Contractions of 16384 and more into many columns
// have a kernel of their own (gemm_kseg.hip) or are the library's.  Over 90 random sizes of 9 to
// 64 rows of 8704 to 16352 into 4112 to 20000 the time here is .89 of the library's, at most
// 1.05 (16 rows of 13824 into 5120 32.7 us there; 8 rows of 14336 into 4096 23.0 us here and
// 24.9, 64 rows 38.2 and 40.2).
static bool linear_few_sizes(long rows, long O, long K) {
  return O >= 1 && K >= 32 && K % 32 == 0 && rows >= 1 && rows <= 64 &&
         !(K >= 16384 && rows > 8 && O > 4096) && !linear_few_other(K);
}

// The same with more rows, where one round of blocks has them all (linear_own.hip).
// O: columns of the result, of two halves of w's rows with a unit.
static bool linear_few_more(long rows, long O, long K, int act) {
  if (rows <= 64) return linear_few_sizes(rows, act ? 2 * O : O, K);
  return !linear_few_other(K) && linear_own_many(rows, O, K, act);
}

// Whether x w^T runs here.
static bool linear_few_takes(const torch::Tensor& x, const torch::Tensor& w) {
  if (!linear_few_input(x) || !linear_few_weight(w, x) || w.size(1) < 1 ||
      x.size(-1) != w.size(1))
    return false;
  return linear_few_sizes(x.numel() / w.size(1), w.size(0), w.size(1));
}

// Whether a product here takes along what it is given: a bias per row of w and norm
// weights per column, side by side, and a residual of the result's shape.  Other forms
// (strides, broadcasts, other types and devices) are those of separate operators.
static bool linear_few_along(const torch::Tensor& x, long O, long biases,
                             const c10::optional<torch::Tensor>& bias,
                             const c10::optional<torch::Tensor>& residual,
                             const c10::optional<torch::Tensor>& norm) {
  auto here = [&](const torch::Tensor& t) {
    return t.device() == x.device() && t.scalar_type() == torch::kBFloat16 &&
           linear_few_plain(t);
  };
  auto vec = [&](const c10::optional<torch::Tensor>& t, long n) {
    return !t.has_value() || (here(*t) && t->is_contiguous() && t->numel() == n);
  };
  // (weights of a norm have to find room in LDS)
  if (!vec(bias, biases) || !vec(norm, x.size(-1)) ||
      (norm.has_value() &&
       (reinterpret_cast<uintptr_t>(norm->data_ptr()) % 16 || x.size(-1) > 32768)))
    return false;
  if (!residual.has_value()) return true;
  return here(*residual) && residual->dim() == x.dim() && residual->size(-1) == O &&
         residual->stride(-1) == 1 &&
         residual->sizes().slice(0, x.dim() - 1) == x.sizes().slice(0, x.dim() - 1);
}

// x's rows, as the kernels read them.
static torch::Tensor linear_few_rows(const torch::Tensor& x) {
  if (x.dim() == 2) return x;
  auto rows = x.reshape({-1, x.size(-1)});
  if (rows.stride(0) % 8 || reinterpret_cast<uintptr_t>(rows.data_ptr()) % 16)
    rows = rows.clone();
  return rows;
}

static torch::Tensor linear_few_shaped(const torch::Tensor& y, const torch::Tensor& x) {
  if (x.dim() == 2) return y;
  auto sizes = x.sizes().vec();
  sizes.back() = y.size(1);
  return y.view(sizes);
}

// Products of more rows (linear_tiles.hip): x [M, K], w [O, K] (act: [2 O, K]).
static torch::Tensor linear_tiles(const torch::Tensor& x, const torch::Tensor& w,
                                  const c10::optional<torch::Tensor>& bias, int64_t act,
                                  int64_t tile, int64_t shares) {
  TORCH_CHECK(linear_few_input(x) && linear_few_weight(w, x) && x.dim() == 2 &&
                  x.size(1) == w.size(1) && act >= 0 && act <= 2 &&
                  linear_few_along(x, w.size(0), w.size(0), bias, {}, {}),
              "linear_tiles takes bf16 rows that begin at multiples of 16 bytes");
  const long M = x.size(0), K = x.size(1), O = w.size(0) / (act ? 2 : 1);
  TORCH_CHECK(M >= 1 && M < 1L << 30 && K % 64 == 0 && O % 64 == 0 && O >= 64 && K < 1L << 22 &&
                  O < 1L << 30 && (!act || (w.size(0) == 2 * O && !bias)) && x.stride(0) >= K &&
                  w.stride(0) >= K && x.stride(0) < 1L << 22 && w.stride(0) < 1L << 22 &&
                  (tile == 128 || tile == 256) && shares >= 1 && (shares == 1 || !act) &&
                  K / 64 / shares >= 3 && shares * M < 1L << 30,
              "sizes that there is no kernel for");
  c10::OptionalDeviceGuard guard;  // and the device's current stream
  if (x.get_device() != c10::hip::current_device()) guard.reset_device(x.device());
  auto y = torch::empty({M, O}, x.options());
  torch::Tensor parts;
  if (bias || shares > 1)
    parts = torch::empty({shares, M, O}, x.options().dtype(torch::kFloat32));
  LinearTilesArgs a{x.data_ptr(), w.data_ptr(), bias ? bias->data_ptr() : nullptr, y.data_ptr(),
                    parts.defined() ? parts.data_ptr<float>() : nullptr, (int)M, (int)O, (int)K,
                    (int)act, (int)shares, x.stride(0) * 2, w.stride(0) * 2};
  launch_linear_tiles(&a, (int)tile, c10::hip::getCurrentHIPStream().stream());
  return y;
}

// (tile, shares) of a product of M rows, tile 0 where it is the library's
static std::pair<int64_t, int64_t> linear_tiles_planned(int64_t M, int64_t O, int64_t K,
                                                        int64_t act, bool bias) {
  int shares = 1;
  const int tile = linear_tiles_plan(M, O, K, (int)act, bias, &shares);
  return {tile, shares};
}

// The product of more than 64 rows, or nothing where it does not run here.
static c10::optional<torch::Tensor> linear_many_try(const torch::Tensor& x,
                                                    const torch::Tensor& w,
                                                    const c10::optional<torch::Tensor>& bias,
                                                    int64_t act) {
  if (w.dim() != 2 || x.dim() < 1 || w.size(1) < 1 || x.size(-1) != w.size(1) ||
      (act && w.size(0) % 2))
    return {};
  const long K = w.size(1), M = x.numel() / K, O = w.size(0) / (act ? 2 : 1);
  if (M <= 64 || M >= 1L << 24) return {};
  const bool own = linear_own_many(M, O, K, (int)act);
  const auto [tile, shares] = own ? std::pair<int64_t, int64_t>{0, 1}
                                  : linear_tiles_planned(M, O, K, act, bias.has_value());
  if ((!own && !tile) || !linear_few_input(x) || !linear_few_weight(w, x) ||
      linear_few_other(K) || !linear_few_along(x, w.size(0), w.size(0), bias, {}, {}))
    return {};
  if (own)
    return linear_few_shaped(
        linear_few_run(linear_few_rows(x), w, bias, {}, {}, 0.0, 0.0, act, {}, {}), x);
  if (w.stride(0) < K || w.stride(0) >= 1L << 22) return {};
  const auto rows = linear_few_rows(x);
  if (rows.stride(0) < K || rows.stride(0) >= 1L << 22) return {};
  return linear_few_shaped(linear_tiles(rows, w, bias, act, tile, shares), x);
}

// linear_few_run for x of any number of dimensions (a product of more rows, on its own:
// linear_tiles), or nothing where it does not run here.
// clear: int32 numbers that are zero afterwards.
static c10::optional<torch::Tensor> linear_few_try(
    torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> bias,
    c10::optional<torch::Tensor> residual, c10::optional<torch::Tensor> norm,
    double eps, double offset, int64_t act, c10::optional<torch::Tensor> clear) {
  if (x.dim() && x.numel() > 64 * x.size(-1)) {
    if (residual.has_value() || norm.has_value() || clear.has_value()) return {};
    return linear_many_try(x, w, bias, act);
  }
  if (!linear_few_takes(x, w) ||
      !linear_few_along(x, w.size(0) / (act ? 2 : 1), w.size(0), bias, residual, norm))
    return {};
  const auto rows = linear_few_rows(x);
  if (residual.has_value() && x.dim() != 2)
    residual = residual->reshape({rows.size(0), -1});
  LinearFewRoom cleared;
  if (clear.has_value()) {
    TORCH_CHECK(clear->device() == x.device() && clear->is_contiguous() &&
                    clear->scalar_type() == torch::kInt32 && clear->numel() < 1 << 20,
                "numbers to clear");
    cleared.numbers = reinterpret_cast<unsigned*>(clear->data_ptr<int>());
    cleared.n = (int)clear->numel();
  }
  return linear_few_shaped(
      linear_few_run(rows, w, bias, residual, norm, eps, offset, act, {}, cleared), x);
}

// The clamped unit of x w^T, with a bias for the first columns of each half, of up to 64 rows and
// of more that linear_own.hip takes, or nothing where that does not run here.
static c10::optional<torch::Tensor> linear_clamped_try(const torch::Tensor& x,
                                                       const torch::Tensor& w,
                                                       const c10::optional<torch::Tensor>& gate,
                                                       const c10::optional<torch::Tensor>& up,
                                                       double limit, double alpha) {
  if (!linear_few_input(x) || !linear_few_weight(w, x) || w.size(1) < 1 || w.size(0) % 2 ||
      x.size(-1) != w.size(1))
    return {};
  const long K = w.size(1), M = x.numel() / K, O = w.size(0) / 2;
  const long n = gate.has_value() ? gate->numel() : O;
  if (linear_few_other(K) || gate.has_value() != up.has_value() || n < 1 || n > O ||
      !linear_few_along(x, O, n, gate, {}, {}) || !linear_few_along(x, O, n, up, {}, {}) ||
      !(M > 64 ? linear_own_many(M, O, K, 3) : linear_few_sizes(M, O, K)))
    return {};
  return linear_few_shaped(
      linear_few_run(linear_few_rows(x), w, gate, {}, {}, limit, alpha, 3, {}, {}, up), x);
}

// A feed-forward: w_out of the gated unit of w_in's halves (act 1 or 2), of x's rows as
// the norm makes them, plus the residual, or nothing where one of the products does not
// run here.  The first clears the numbers that the blocks of the second count with.
static c10::optional<torch::Tensor> feed_few_try(
    torch::Tensor x, torch::Tensor w_in, torch::Tensor w_out,
    c10::optional<torch::Tensor> residual, c10::optional<torch::Tensor> norm, double eps,
    double offset, int64_t act) {
  TORCH_CHECK(act == 1 || act == 2, "unknown unit");
  if (!linear_few_input(x) || !linear_few_weight(w_in, x) || !linear_few_weight(w_out, x) ||
      w_in.size(1) < 1 || x.size(-1) != w_in.size(1) || w_in.size(0) != 2 * w_out.size(1) ||
      !linear_few_more(x.numel() / w_in.size(1), w_out.size(1), w_in.size(1), (int)act))
    return {};
  const int M = x.numel() / x.size(-1), O = w_out.size(0), I = w_out.size(1);
  // long contractions into many columns have a kernel of their own (gemm_kseg.hip)
  if (I >= 16384 && O >= 8192 && !residual.has_value()) return {};
  if (!linear_few_more(M, O, I, 0) ||
      !linear_few_along(x, I, 2 * I, {}, {}, norm) ||
      !linear_few_along(x, O, O, {}, residual, {}))
    return {};
  const auto rows = linear_few_rows(x);
  if (residual.has_value() && x.dim() != 2) residual = residual->reshape({M, -1});
  const auto room = M <= 64 ? LinearFewRoom(M, O, I, rows) : LinearFewRoom();
  const auto units =
      linear_few_run(rows, w_in, {}, {}, norm, eps, offset, act, {}, room);
  return linear_few_shaped(
      linear_few_run(units, w_out, {}, residual, {}, 0.0, 0.0, 0, room, {}), x);
}
