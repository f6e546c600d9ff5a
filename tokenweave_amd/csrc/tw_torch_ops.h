// What tw_torch_binding.cpp registers with torch's dispatcher, callable from C++ as well: the
// Python module of direct calls (tw_hostpath.cpp) goes straight to these functions.  Each
// checks its arguments (c10::Error on a bad one, before anything is enqueued) and enqueues one
// kernel on the current stream of the tensors' device.
#ifndef TW_TORCH_OPS_H
#define TW_TORCH_OPS_H

#include <ATen/ATen.h>

#include <optional>
#include <vector>

#define TW_TORCH_API __attribute__((visibility("default")))

namespace tw_torch {

using at::Tensor;

TW_TORCH_API void rms_norm(Tensor& out, Tensor& input, Tensor& weight, double epsilon);
TW_TORCH_API void fused_add_rms_norm(Tensor& input, Tensor& residual, Tensor& weight, double epsilon);
TW_TORCH_API void rms_norm_inplace(Tensor& out, Tensor& input, Tensor& weight, double epsilon);
TW_TORCH_API void fused_add_rms_norm_cta(Tensor& input, Tensor& residual, Tensor& weight, int64_t max_ctas,
                                         double epsilon);
// Rows [row0, row0 + rows) of `input` and `residual`; `mcptr` addresses row `row0` in slot 0.
TW_TORCH_API void fused_rs_ln_rows(bool all_gather, const Tensor& input, const Tensor& residual, const Tensor& weight,
                                   int64_t row0, int64_t rows, int64_t mcptr, int64_t rank, int64_t world_size,
                                   int64_t max_ctas, double epsilon);
TW_TORCH_API void rms_norm_static_fp8_quant(Tensor& out, Tensor& input, Tensor& weight, Tensor& scale, double epsilon);
TW_TORCH_API void fused_add_rms_norm_static_fp8_quant(Tensor& out, Tensor& input, Tensor& residual, Tensor& weight,
                                                      Tensor& scale, double epsilon);
TW_TORCH_API void rms_norm_dynamic_per_token_quant(Tensor& out, const Tensor& input, const Tensor& weight,
                                                   Tensor& scales, double epsilon, std::optional<Tensor> scale_ub,
                                                   std::optional<Tensor> residual);
// out[M, N] <- a[M, K] b[N, K]^T (+ bias, added to the rounded product); not registered: no
// reference schema.  `bias` may be null.
TW_TORCH_API void gemm_bf16_nt(const Tensor& out, const Tensor& a, const Tensor& b, int64_t max_cus,
                               const Tensor* bias);
// One launch for several products of one shape; `biases` is empty or has an entry (maybe null)
// for each.
TW_TORCH_API void gemm_bf16_nt_partials(const std::vector<const Tensor*>& outs, const std::vector<const Tensor*>& a,
                                        const std::vector<const Tensor*>& b, int64_t max_cus,
                                        const std::vector<const Tensor*>& biases);

}  // namespace tw_torch

#endif
