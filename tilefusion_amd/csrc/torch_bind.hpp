// The op implementations of torch_bind.cc, for direct_call.cc.
#pragma once

#include <ATen/ATen.h>

#include <cstdint>

namespace tilefusion::kernels {

extern "C" {
void gemm(const at::Tensor& A, const at::Tensor& B, at::Tensor& C, int64_t tm, int64_t tn, int64_t tk,
          int64_t num_stages, int64_t pipeline_level);
void fused_two_gemms(const at::Tensor& A, const at::Tensor& B, const at::Tensor& C, at::Tensor& D, int64_t tm,
                     int64_t tn, int64_t tk, int64_t tp);
void scatter_nd(const at::Tensor& data, at::Tensor& updates, const at::Tensor& indices);
}
void flash_attention_fwd(const at::Tensor& Q, const at::Tensor& K, const at::Tensor& V, at::Tensor& O,
                         double softmax_scale, bool causal);
void flash_attention_fwd_kt(const at::Tensor& Q, const at::Tensor& K, const at::Tensor& V, at::Tensor& O,
                            double softmax_scale, bool causal);
void flash_decode(const at::Tensor& Q, const at::Tensor& K, const at::Tensor& V, at::Tensor& O, int64_t num_splits,
                  double softmax_scale);

}  // namespace tilefusion::kernels
