// gptq::linear_rows, the dequant-GEMV/GEMM entry point as a native torch
// operator: what a decode step calls once per layer, where a Python
// implementation (operator wrapper, argument checks, ctypes marshalling) took
// 25 us around kernels of 5-15 us.  The caller has resolved the layer's
// layout (code width, contiguous groups); autograd and layouts with a group
// index go through gptq::linear.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>

#include "gptq_hip.h"

namespace {

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return GPTQ_F32;
    case at::kHalf: return GPTQ_F16;
    case at::kBFloat16: return GPTQ_BF16;
    default: TORCH_CHECK_TYPE(false, "unsupported dtype ", t, "; expected float32, float16 or bfloat16");
  }
}

// y = x @ dequant(W)^T (+ bias), x (..., K): as gptq_linear_ws, on x's current stream
at::Tensor linear_rows(const at::Tensor& x, const at::Tensor& qweight, const at::Tensor& scales,
                       const at::Tensor& zeros, const std::optional<at::Tensor>& bias,
                       const std::optional<at::Tensor>& perm, int64_t bits, int64_t group_size, int64_t K) {
  // what is refused is a ValueError or a TypeError, which the caller leaves to
  // gptq::linear; everything else is a failure
  TORCH_CHECK_VALUE(x.is_cuda() && qweight.device() == x.device() && scales.device() == x.device() &&
                        zeros.device() == x.device() && (!bias || bias->device() == x.device()) &&
                        (!perm || perm->device() == x.device()),
                    "gptq::linear_rows: expected GPU tensors on one device");
  TORCH_CHECK_VALUE(K > 0 && x.dim() > 0 && x.size(-1) == K && qweight.dim() == 2 && scales.dim() == 2 &&
                        zeros.sizes() == scales.sizes() && scales.size(0) == qweight.size(0) &&
                        qweight.scalar_type() == at::kByte && qweight.is_contiguous() &&
                        qweight.size(1) == (bits == 0 ? K : (K * bits + 7) / 8) &&
                        (!bias || bias->numel() == qweight.size(0)),
                    "gptq::linear_rows: the shapes of x and the weight do not match in_features = ", K);
  const c10::DeviceGuard guard(x.device());
  const int64_t N = qweight.size(0);
  const at::Tensor x2 = x.reshape({-1, K}).contiguous();
  const int64_t M = x2.size(0);
  const at::Tensor s = scales.contiguous(), z = zeros.to(scales.scalar_type()).contiguous();
  at::Tensor b, p;
  if (bias) b = bias->contiguous();
  if (perm) {
    TORCH_CHECK_VALUE(perm->numel() == K, "perm has ", perm->numel(), " entries, in_features is ", K);
    p = perm->to(at::kInt).contiguous();
  }
  const int xt = dtype_code(x2.scalar_type());
  std::vector<int64_t> shape = x.sizes().vec();
  shape.back() = N;
  at::Tensor y = at::empty(shape, x2.options());
  // exactly the requested size, so that the kernel choice depends on the
  // shapes only; from the caching allocator, ordered on this stream
  const size_t bytes = gptq_linear_workspace_size(M, N, K, static_cast<int>(bits), static_cast<int>(group_size), xt, perm ? 1 : 0);
  at::Tensor ws;
  if (bytes) ws = at::empty({static_cast<int64_t>(bytes)}, x2.options().dtype(at::kByte));
  const int rc = gptq_linear_ws(
      x2.const_data_ptr(), xt, M, perm ? p.const_data_ptr<int32_t>() : nullptr, qweight.const_data_ptr<uint8_t>(),
      static_cast<int>(bits), s.const_data_ptr(), z.const_data_ptr(), dtype_code(s.scalar_type()), nullptr,
      static_cast<int>(group_size), s.size(1), bias ? b.const_data_ptr() : nullptr,
      bias ? dtype_code(b.scalar_type()) : 0, N, K, y.mutable_data_ptr(), bytes ? ws.mutable_data_ptr() : nullptr, bytes,
      c10::hip::getCurrentHIPStream(x.device().index()).stream());
  TORCH_CHECK_VALUE(rc != GPTQ_ERR_ARG && rc != GPTQ_ERR_SHAPE, "gptq_linear_ws: ", gptq_last_error());
  TORCH_CHECK_TYPE(rc != GPTQ_ERR_DTYPE, "gptq_linear_ws: ", gptq_last_error());
  TORCH_CHECK(rc == GPTQ_OK, "gptq_linear_ws failed (status ", rc, "): ", gptq_last_error());
  return y;
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(gptq, m) {
  m.def("linear_rows(Tensor x, Tensor qweight, Tensor scales, Tensor zeros, Tensor? bias, Tensor? perm, int bits, "
        "int group_size, int in_features) -> Tensor");
}

TORCH_LIBRARY_IMPL(gptq, CUDA, m) { m.impl("linear_rows", linear_rows); }
