// Shared by the FP32 prefill GEMMs (gemm_f32.hip, gemm_chain.hip): arguments
// and the epilogue.
#pragma once

#include "focr_internal.hpp"

namespace focr {

struct GemmArgs {
  const float *x;
  const float *row_scale;
  const void *codes;
  const float *scales;
  const int16_t *exc_index;
  const int32_t *exc_cols;
  const float *exc_vals;
  int n_exc;
  int m, n, k, group, groups;
  float *out;
  int row0;  // dma_kernel: first output row of the launch's tiles (0 for the other kernels)
};

// The exact-order GEMM on the FP32 matrix cores (gemm_chain.hip); false, and
// nothing launched, for the shapes it does not take.
bool launch_chain_mfma(const GemmArgs &a, int bits, int epilogue, hipStream_t stream);

// Writes one output value through the epilogue. For GLU, `partner` is the
// value of the neighbouring column (col ^ 1), fetched by the caller.
template <int EPI>
__device__ __forceinline__ void emit(const GemmArgs &a, int row, int col, float v, float partner) {
  if (row >= a.m || col >= a.n) return;
  if constexpr (EPI == FOCR_EPI_GLU) {
    if ((col & 1) == 0) a.out[static_cast<size_t>(row) * (a.n / 2) + col / 2] = squared_relu_glu(v, partner);
  } else if constexpr (EPI == FOCR_EPI_ADD) {
    float *dst = a.out + static_cast<size_t>(row) * a.n + col;
    *dst = *dst + v;
  } else {
    a.out[static_cast<size_t>(row) * a.n + col] = v;
  }
}

}  // namespace focr
