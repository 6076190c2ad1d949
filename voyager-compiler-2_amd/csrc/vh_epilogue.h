// The GEMM epilogue of one float32 accumulator (vh_epilogue), shared by the
// GEMM kernels.
#pragma once

#include "vh_device.h"

namespace {

__device__ __forceinline__ float epi_scale(const vh_epilogue& e) {
  if (!e.scale) return 1.0f;
  return e.scale_dtype == VH_BF16 ? bf2f(*(const uint16_t*)e.scale) : *(const float*)e.scale;
}

__device__ __forceinline__ float epi_bias(const vh_epilogue& e, int64_t col) {
  if (!e.bias) return 0.0f;
  return e.bias_dtype == VH_BF16 ? bf2f(((const uint16_t*)e.bias)[col]) : ((const float*)e.bias)[col];
}

// The epilogue of one fp32 accumulator (sc = epi_scale, bias = epi_bias).
__device__ __forceinline__ float epi_value(const vh_epilogue& e, float v, float sc, float bias) {
  if (e.mode == EPI_ROUND_SCALE) {
    // dequantize(linear(xq, wq), s): the GEMM rounds to bf16, then the bf16
    // product with the scale rounds again.
    return rbf(rbf(v) * sc);
  }
  if (e.scale) v = v * sc;
  if (e.bias) v = v + bias;
  return v;
}

}  // namespace
