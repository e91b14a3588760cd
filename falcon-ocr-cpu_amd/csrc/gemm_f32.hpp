// Shared by the FP32 prefill GEMMs (gemm_f32.hip, gemm_chain.hip): arguments,
// the epilogue, the LDS-DMA types and waits, the tile order.
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

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void global_void;

// s_waitcnt immediate for vmcnt(n) (n < 64) and lgkmcnt(0), expcnt not waited.
constexpr int wait_vm_lgkm0(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0070; }

// Compiler-only ordering around the plain workgroup barrier: the waits are
// explicit (a __syncthreads fence would wait for every copy in flight).
__device__ __forceinline__ void plain_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Tile order: workgroups are dealt to the 8 XCDs round robin (block b runs on
// XCD b % 8); block b takes tile t = (b % 8) * per + b / 8, so each XCD walks
// a contiguous run of tiles, in panels of kTilePanel row tiles (column tiles
// in order, rows fastest): the workgroups an XCD holds at once share a few A
// row tiles and B column tiles in its own L2.
constexpr int kTilePanel = 4;
__device__ __forceinline__ void xcd_tile(int b, int row_tiles, int col_tiles, int &rt, int &ct) {
  const int total = row_tiles * col_tiles;
  const int per = total / 8;
  const int t = b < 8 * per ? (b % 8) * per + b / 8 : b;
  const int panel = t / (kTilePanel * col_tiles);
  const int rem = t - panel * kTilePanel * col_tiles;
  const int rows = row_tiles - panel * kTilePanel < kTilePanel ? row_tiles - panel * kTilePanel : kTilePanel;
  ct = rem / rows;
  rt = panel * kTilePanel + rem % rows;
}


}  // namespace focr
