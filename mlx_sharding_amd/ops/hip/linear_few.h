// y = x W^T for up to 64 rows, with what goes with it (linear_few.hip); part of
// both extensions.
#pragma once

#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

extern "C" void launch_linear_few(const void*, const void*, const void*,
                                  const void*, const void*, void*, int, int, int,
                                  long, long, long, long, float, float, int,
                                  hipStream_t);

// x [M, K], w [O, K] (act: [2 O, K]); bias per row of w, residual [M, O], norm
// weights [K] for the rows of x; act 0: none, 1: silu, 2: gelu_tanh
static torch::Tensor linear_few(torch::Tensor x, torch::Tensor w,
                                c10::optional<torch::Tensor> bias,
                                c10::optional<torch::Tensor> residual,
                                c10::optional<torch::Tensor> norm, double eps,
                                double offset, int64_t act) {
  auto bf16 = [](const torch::Tensor& t) {
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kBFloat16,
                "linear_few takes bf16 tensors on the GPU");
  };
  auto whole = [](const torch::Tensor& t) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  bf16(x);
  bf16(w);
  TORCH_CHECK(act >= 0 && act <= 2, "unknown unit");
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1), "shapes");
  const int M = x.size(0), K = x.size(1), O = w.size(0) / (act ? 2 : 1);
  TORCH_CHECK(M >= 1 && M <= 64 && K >= 32 && K % 32 == 0 && O >= 1,
              "1 to 64 rows of a multiple of 32");
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
  const void* b = vec(bias, w.size(0));
  const void* n = vec(norm, K);
  TORCH_CHECK(!n || whole(*norm), "norm weights begin at a multiple of 16 bytes");
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
  auto y = torch::empty({M, O}, x.options());
  launch_linear_few(x.data_ptr(), w.data_ptr(), b, r, n, y.data_ptr(), M, O, K,
                    x.stride(0), w.stride(0), ldr, O, (float)eps, (float)offset,
                    (int)act, c10::hip::getCurrentHIPStream().stream());
  return y;
}
