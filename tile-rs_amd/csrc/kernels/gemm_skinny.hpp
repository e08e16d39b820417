// 16-bit GEMM with few rows of A (M up to 64: the projections of a decode step), B stored
// N x K.
//
// Bound: HBM, the one read of B.  No split of K over workgroups, so no partials and no
// second launch: a workgroup owns 16 NF columns, its four waves take quarters of K and their
// f32 sums are added through LDS, in wave order, at the end.  Each wave streams its quarter
// through an LDS ring of its own (R stages of 64 k), so the loop has no barrier: wait for
// the oldest stage's DMA, read its fragments, multiply, refill the stage.  A stage is 16 NF
// rows of B and XR rows of A, 128 bytes each, fetched as whole lines (eight rows per DMA;
// register loads of MFMA fragments, 64 bytes of 16 rows, ran 26 us where this takes 21),
// 16-byte chunk c of row r at c ^ (r % 8).  B is the MFMA's first operand, so D = B A^T and
// lanes hold consecutive columns of a row of C.
//
// Every workgroup reads all of A (from L2), so NF grows with N while the grid still fills the
// chip, and A's re-reads bound the rule in ops_gemm_skinny.hip.  Rows past M (columns past
// N) read the last row and are not stored.
//
// Measured on MI355X against the split-K kernel and its merge (bf16): 8 x 14336 x 4096
// 27.2 -> 21.3 us (5.5 TB/s), 16 x 4096 x 14336 29 -> 24, 8 x 4096 x 4096 12 -> 7.5,
// 64 x 4096 x 4096 15.2 -> 10.8, 16 x 4096 x 1024 9.9 -> 6.0.
#pragma once

#include "gemm.hpp"

namespace th {
namespace gskinny {
constexpr int WAVES = 4;
constexpr int NT = 64 * WAVES;
constexpr int KU = 64;      // K per stage
constexpr int kMaxM = 64;

// Stages of the ring: 3 workgroups per CU at the smallest shape, 1 at the largest (the
// fastest of 2 to 8 measured for each).
template <int XR, int NF>
constexpr int kStages = NF == 1 ? (XR == 64 ? 3 : 4) : NF == 2 ? (XR == 8 ? 4 : 3) : (XR == 32 ? 3 : 2);
}  // namespace gskinny

// Columns [n0, n0 + 16 NF) of C = epilogue(A . B^T), M <= XR rows.  K % 8 == 0, A and B
// 16-byte aligned.
template <int DT, int DT_OUT, int EPI, int XR, int NF>
__device__ __forceinline__ void gemm_skinny_tile(const uint16_t* __restrict__ A,
                                                 const uint16_t* __restrict__ B,
                                                 void* __restrict__ C, uint32_t M, uint32_t N,
                                                 uint32_t K, uint32_t n0,
                                                 const void* __restrict__ up) {
  using namespace gskinny;
  static_assert(XR == 8 || XR == 16 || XR == 32 || XR == 64, "rows");
  constexpr int R = kStages<XR, NF>;
  constexpr int NB = 2 * NF, ND = NB + XR / 8;   // DMAs per stage: B, then A
  constexpr int MT = (XR + 15) / 16;             // 16-row blocks of A
  constexpr int ST = 64 * ND;                    // 16-byte slots per stage
  u32x4* arena = lds::dma_lds_arena<WAVES * R * ST * 16>();
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  u32x4* ring = arena + wave * R * ST;

  // this wave's stages; the last wave also takes the K % 64 values after them
  const uint32_t units = K / KU, per = (units + WAVES - 1) / WAVES;
  const uint32_t u0 = min(units, wave * per), n = min(units, u0 + per) - u0;

  // DMA: lane l fills slot l % 8 of row l / 8 of its eight
  const int r8 = lane >> 3, chunk = 8 * ((lane & 7) ^ r8);
  const uint16_t* src[ND];
#pragma unroll
  for (int j = 0; j < ND; ++j) {
    const uint16_t* base = j < NB ? B + static_cast<size_t>(min(n0 + 8 * j + r8, N - 1)) * K
                                  : A + static_cast<size_t>(min(8u * (j - NB) + r8, M - 1)) * K;
    src[j] = base + chunk + u0 * KU;
  }
  // stages past the last re-read it, so that the count in flight stays the same
  auto issue = [&](uint32_t i) {
    const size_t k = static_cast<size_t>(min(i, n - 1)) * KU;
    u32x4* d = ring + (i % R) * ST;
#pragma unroll
    for (int j = 0; j < ND; ++j) lds::dma16(src[j] + k, d + 64 * j);
  };

  f32x4 acc[NF][MT];
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[f][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  if (n > 0) {
#pragma unroll
    for (int i = 0; i < R; ++i) issue(i);
    // fragments: lane l reads row l % 16 at k 8 (l / 16) .. +7 of each 32
    const int c0 = g ^ (l16 & 7), c1 = (4 + g) ^ (l16 & 7);
    for (uint32_t i = 0; i < n; ++i) {
      lds::wait_vm<(R - 1) * ND>();
      asm volatile("" ::: "memory");
      const u32x4* s = ring + (i % R) * ST;
      u32x4 b[NF][2], a[MT][2];
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        b[f][0] = s[(16 * f + l16) * 8 + c0];
        b[f][1] = s[(16 * f + l16) * 8 + c1];
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int row = XR == 8 ? (l16 & 7) : 16 * m + l16;
        a[m][0] = s[64 * NB + row * 8 + c0];
        a[m][1] = s[64 * NB + row * 8 + c1];
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[f][m] = mfma16x16x32<DT>(b[f][h], a[m][h], acc[f][m]);
      lds::wait_lgkm0();   // the stage is read
      asm volatile("" ::: "memory");
      issue(i + R);
    }
    lds::wait_vm<0>();
  }
  if (wave == WAVES - 1) {
    for (uint32_t k0 = units * KU; k0 < K; k0 += 32) {
      const uint32_t k = k0 + 8 * g;
      const u32x4 zero = {0, 0, 0, 0};
      u32x4 a[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m)
        a[m] = k < K ? ldg128(A + static_cast<size_t>(min(16u * m + l16, M - 1)) * K + k) : zero;
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const u32x4 b =
            k < K ? ldg128(B + static_cast<size_t>(min(n0 + 16 * f + l16, N - 1)) * K + k) : zero;
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[f][m] = mfma16x16x32<DT>(b, a[m], acc[f][m]);
      }
    }
  }

  // Sum over the waves: D's column l % 16 is row m of C, its row 4 (l / 16) + r column
  // 4 (l / 16) + r of block f.
  static_assert(WAVES * NF * MT * 64 <= WAVES * R * ST, "reduction space");
  __syncthreads();
  float* red = reinterpret_cast<float*>(arena);
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int m = 0; m < MT; ++m)
      *reinterpret_cast<f32x4*>(&red[((wave * NF * MT + f * MT + m) * 64 + lane) * 4]) = acc[f][m];
  __syncthreads();
  for (int o = t; o < 256 * NF * MT; o += NT) {
    const int col = o % (16 * NF), m = o / (16 * NF), i = col & 15;
    const float* p = &red[(((col >> 4) * MT + (m >> 4)) * 64 + 16 * (i >> 2) + (m & 15)) * 4 + (i & 3)];
    float v = p[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) v += p[w * NF * MT * 256];
    if (m < static_cast<int>(M) && n0 + col < N)
      gemm::store_out<EPI, DT_OUT>(C, up, static_cast<size_t>(m) * N + n0 + col, v);
  }
}

// Grid: x = ceil(N / (16 NF)), y = batch (element strides sa, sb, sc).
template <int DT, int DT_OUT, int EPI, int XR, int NF>
__global__ void __launch_bounds__(gskinny::NT)
gemm_skinny(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B, void* __restrict__ C,
            uint32_t M, uint32_t N, uint32_t K, uint64_t sa, uint64_t sb, uint64_t sc,
            const void* __restrict__ up) {
  constexpr int OSZ = (DT_OUT == kF32) ? 4 : 2;
  const size_t co = static_cast<size_t>(blockIdx.y) * sc * OSZ;
  gemm_skinny_tile<DT, DT_OUT, EPI, XR, NF>(A + blockIdx.y * sa, B + blockIdx.y * sb,
                                            static_cast<char*>(C) + co, M, N, K,
                                            blockIdx.x * 16 * NF,
                                            up ? static_cast<const char*>(up) + co : nullptr);
}

}  // namespace th
