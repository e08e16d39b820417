// Shared by the GEMM translation units (ops_gemm.hip: entry points and 16-bit operands;
// ops_gemm_skinny.hip: 16-bit operands with few rows; ops_gemm_f32.hip: f32 operands).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "ops_common.hpp"

namespace th {
namespace ops {

// One GEMM launch: C[i] = epilogue(A[i] . B[i]) for i < batch, element strides
// sa, sb, sc; `up` (epilogue kEpiSiluMul) has C's dtype, layout and strides.
struct GemmArgs {
  const void* a;
  const void* b;
  void* c;
  const void* up;
  uint32_t m, k, n;
  bool bt;
  uint32_t batch;
  uint64_t sa, sb, sc;
  hipStream_t s;
  uint32_t slices = 1;   // K slices of the 256 x 256 LDS-DMA kernel
};

// C = epilogue(sum of the S partials of M x N f32 at W, in ascending order).
int splitk_merge(const GemmArgs& g, const float* W, uint32_t S, th_dtype out, int epi);

// f32 operands.
int gemm_f32(const GemmArgs& g, th_dtype out, int epi);

// 16-bit operands, few rows of A, B stored N x K: whether the kernel is the one for the
// shape, and its launch (K % 8 == 0, A and B and their strides 16-byte aligned).
bool few_rows_fit(const GemmArgs& g);
int gemm_few_rows(const GemmArgs& g, th_dtype in, th_dtype out, int epi);

// The form of a 16-bit product (the same conditions): tile, K slices and their depth.
struct GemmPlan {
  enum { k64x64, k128x64, k256 };
  int tile;
  uint32_t slices, ks;
  bool in_graph;   // split while a graph is recorded as well
};
// What the 256 x 256 kernels can do with it: the assembly kernel (whole), the LDS-DMA kernel
// (dma; else the register-staged one), and the K split of the latter (1: none).
struct GemmForms {
  bool whole, dma;
  uint32_t split;
};
GemmPlan plan_16bit(const GemmArgs& g, const GemmForms& f);
int gemm_mid_tiles(const GemmArgs& g, th_dtype in, th_dtype out, int epi, const GemmPlan& p);

}  // namespace ops
}  // namespace th
