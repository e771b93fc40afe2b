// Column sums as an op (sxe_colsum.h): the bias gradients of linear layers and of the bias + activation kernels. The reference sums
// with torch (module_inject / runtime autograd); its fused transformer layer has a column reduction of its own
// (csrc/transformer/general_kernels.cu).
#include "sxe_colsum.h"
#include <torch/library.h>

namespace sxe {

// x [R, N] with unit column stride (any row stride), bf16 / f16 / fp32 -> [N] of `dtype`: that of x, or fp32
at::Tensor column_sum(const at::Tensor& x, at::ScalarType dtype) {
  SXE_CHECK_CUDA(x);
  SXE_CHECK(x.dim() == 2 && (x.stride(1) == 1 || x.size(1) <= 1), "column_sum: [R, N] with unit column stride");
  SXE_CHECK(dtype == x.scalar_type() || dtype == at::kFloat, "column_sum: the result is of x's type or fp32");
  const int64_t R = x.size(0), N = x.size(1);
  c10::DeviceGuard gd(x.device());
  if (R == 0 || N == 0) return at::zeros({N}, x.options().dtype(dtype));
  auto out = at::empty({N}, x.options().dtype(dtype));
  const void* const in[2] = {x.data_ptr(), nullptr};
  void* const o[2] = {out.data_ptr(), nullptr};
  auto go = [&](auto t) {
    constexpr DT T = decltype(t)::value;
    if (dtype == at::kFloat) colsum<T, DT::F32>(in, o, R, N, x.stride(0), 1, x.options());
    else colsum<T, T>(in, o, R, N, x.stride(0), 1, x.options());
  };
  switch (dtype_of(x)) {
    case DT::F32: go(std::integral_constant<DT, DT::F32>{}); break;
    case DT::BF16: go(std::integral_constant<DT, DT::BF16>{}); break;
    case DT::F16: go(std::integral_constant<DT, DT::F16>{}); break;
  }
  return out;
}

// out fp32 [N] = [out +] the column sums of x
void column_sum_(const at::Tensor& x, at::Tensor out, bool accumulate) {
  check_beside(x, {out});
  SXE_CHECK(x.dim() == 2 && (x.stride(1) == 1 || x.size(1) <= 1) && out.scalar_type() == at::kFloat && out.is_contiguous() &&
                out.numel() == x.size(1), "column_sum_: [R, N] with unit column stride, fp32 out [N]");
  const int64_t R = x.size(0), N = x.size(1);
  c10::DeviceGuard gd(x.device());
  if (R == 0 || N == 0) {
    if (!accumulate) out.zero_();
    return;
  }
  const void* const in[2] = {x.data_ptr(), nullptr};
  void* const o[2] = {out.data_ptr(), nullptr};
  auto go = [&](auto t) { colsum<decltype(t)::value, DT::F32>(in, o, R, N, x.stride(0), 1, x.options(), accumulate); };
  switch (dtype_of(x)) {
    case DT::F32: go(std::integral_constant<DT, DT::F32>{}); break;
    case DT::BF16: go(std::integral_constant<DT, DT::BF16>{}); break;
    case DT::F16: go(std::integral_constant<DT, DT::F16>{}); break;
  }
}

}  // namespace sxe

TORCH_LIBRARY_FRAGMENT(sxe, m) {
  m.def("column_sum(Tensor x, ScalarType dtype) -> Tensor");
  m.def("column_sum_(Tensor x, Tensor(a!) out, bool accumulate) -> ()");
}
TORCH_LIBRARY_IMPL(sxe, CUDA, m) {
  m.impl("column_sum", &sxe::column_sum);
  m.impl("column_sum_", &sxe::column_sum_);
}
