// f32 GEMM on gfx950's fp32 matrix cores (v_mfma_f32_32x32x2_f32): the
// __tile_matmul_f32 op (crates/tile_std/src/tile.rs:193, :2309; linalg
// semantics crates/rustc_codegen_tile/src/mlir_to_linalg.rs:1345-1393: C = A.B
// with f32 accumulation).
//
// One 128 x 128 tile of C per 256-thread workgroup: 2 x 2 waves, each 64 x 64 =
// 2 x 2 blocks of 32 x 32 accumulators (64 registers).  K advances 16 at a time
// through two LDS buffers.  Both operands sit in LDS k-major, A^T[k][m] and
// B[k][n], because the MFMA's two k values per step go to the two lane halves
// (lane l holds A[m = l % 32][k = l / 32] and B[k = l / 32][n = l % 32]): every
// operand fetch is one 4-byte LDS read of 32 consecutive values per half.  Rows
// are 128 + 32 floats long so that rows k and k + 1 fall in opposite halves of
// the 64 banks.  A (and B^T when B is given as N x K) is transposed on its way
// into LDS; row-major B is copied as is.  The next K step's tiles are loaded
// into registers while the current one computes (one barrier per step).
//
// The MFMA multiplies and adds in f32 (no reduced-precision inputs); only the
// order of the K sum differs from a sequential FMA loop.
#pragma once

#include "common.hpp"
#include "gemm.hpp"

namespace th {
namespace gf32 {
constexpr int BM = 128, BN = 128, BK = 16;
// Tile-rows per XCD group.  Four workgroups per CU run an XCD's whole run of
// tiles at once (128 at 4096^3); groups 8 tall make that run 8 x 16 tiles, which
// reads 8 A and 16 B panels instead of 4 and 32 (groups 4 tall).
constexpr int GROUP_M = 8;
constexpr int LD = 128 + 32;  // LDS row (floats)
constexpr int NT = 256;

typedef float f32x16 __attribute__((ext_vector_type(16)));

// 16-byte aligned: row-major B tiles go in with 16-byte LDS writes
struct alignas(16) Lds {
  float a[2][BK * LD];
  float b[2][BK * LD];
};
__device__ __forceinline__ Lds& smem() {
  __shared__ Lds s;
  return s;
}

// 4 consecutive floats of row `r` (`cols` long, row stride `ld`) from column c,
// zero past the matrix; one 16-byte load when VEC and the 4 are in range.
template <bool VEC>
__device__ __forceinline__ f32x4 load4(const float* __restrict__ p, uint32_t r, uint32_t c,
                                       uint32_t rows, uint32_t cols, size_t ld) {
  f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
  if (r >= rows) return v;
  const float* q = p + static_cast<size_t>(r) * ld + c;
  if (VEC && c + 4 <= cols) return *reinterpret_cast<const f32x4*>(q);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (c + j < cols) v[j] = q[j];
  return v;
}
}  // namespace gf32

// Tile (tm, tn) of C (M x N, row stride N) = A (M x K) . B (K x N, or N x K when
// B_TRANS).  VEC: every row start of A and B is 16-byte aligned (K % 4 == 0 and,
// for row-major B, N % 4 == 0, aligned bases), so full 4-float pieces load as one.
template <int DT_OUT, bool B_TRANS, bool VEC, int EPI>
__device__ __forceinline__ void gemm_f32_tile_128(const float* __restrict__ A,
                                                  const float* __restrict__ B,
                                                  void* __restrict__ C, uint32_t M, uint32_t N,
                                                  uint32_t K, uint32_t tm, uint32_t tn,
                                                  const void* __restrict__ up) {
  using namespace gf32;
  Lds& s = smem();
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const uint32_t m0 = tm * BM, n0 = tn * BN;

  // staging: A piece i covers rows (t + 256 i) % 128, k (t + 256 i) / 128 * 4 ..+3,
  // so the 64 lanes of a wave write 64 consecutive m of one A^T row.
  constexpr int NP = BM * BK / 4 / NT;   // 16-byte pieces per thread per operand
  f32x4 ra[NP], rb[NP];
  auto load = [&](uint32_t k0) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int e = t + 256 * i;
      ra[i] = load4<VEC>(A, m0 + (e & 127), k0 + (e >> 7) * 4, M, K, K);
      if constexpr (B_TRANS) rb[i] = load4<VEC>(B, n0 + (e & 127), k0 + (e >> 7) * 4, N, K, K);
      else rb[i] = load4<VEC>(B, k0 + (e >> 5), n0 + (e & 31) * 4, K, N, N);
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int e = t + 256 * i;
      const int r = e & 127, k4 = (e >> 7) * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) s.a[buf][(k4 + j) * LD + r] = ra[i][j];
      if constexpr (B_TRANS) {
#pragma unroll
        for (int j = 0; j < 4; ++j) s.b[buf][(k4 + j) * LD + r] = rb[i][j];
      } else {
        *reinterpret_cast<f32x4*>(&s.b[buf][(e >> 5) * LD + (e & 31) * 4]) = rb[i];
      }
    }
  };

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  const int h = lane >> 5, l32 = lane & 31;
  const int ao = wm * 64 + l32, bo = wn * 64 + l32;
  const uint32_t nk = (K + BK - 1) / BK;
  load(0);
  store(0);
  __syncthreads();
  for (uint32_t kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < nk) load((kt + 1) * BK);
    const float* sa = s.a[cur] + h * LD + ao;
    const float* sb = s.b[cur] + h * LD + bo;
#pragma unroll
    for (int ks = 0; ks < BK / 2; ++ks) {
      const float a0 = sa[2 * ks * LD], a1 = sa[2 * ks * LD + 32];
      const float b0 = sb[2 * ks * LD], b1 = sb[2 * ks * LD + 32];
      acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b0, acc[0][0], 0, 0, 0);
      acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b1, acc[0][1], 0, 0, 0);
      acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b0, acc[1][0], 0, 0, 0);
      acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b1, acc[1][1], 0, 0, 0);
    }
    if (kt + 1 < nk) store(cur ^ 1);
    __syncthreads();
  }

  // accumulator r of a 32 x 32 block: row 8 (r / 4) + 4 h + r % 4, column l32
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint32_t col = n0 + wn * 64 + 32 * j + l32;
      if (col >= N) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t row = m0 + wm * 64 + 32 * i + 8 * (r >> 2) + 4 * h + (r & 3);
        if (row < M)
          gemm::store_out<EPI, DT_OUT>(C, up, static_cast<size_t>(row) * N + col, acc[i][j][r]);
      }
    }
}

// Library kernel: tiles in XCD-aware grouped order (GROUP_M), batch = blockIdx.y with
// element strides sa, sb, sc.
template <int DT_OUT, bool B_TRANS, bool VEC, int EPI = 0>
__global__ void __launch_bounds__(gf32::NT)
gemm_f32_mfma(const float* __restrict__ A, const float* __restrict__ B, void* __restrict__ C,
              uint32_t M, uint32_t N, uint32_t K, uint64_t sa, uint64_t sb, uint64_t sc,
              const void* __restrict__ up) {
  constexpr int OSZ = (DT_OUT == kF32) ? 4 : 2;
  const uint32_t tiles_m = (M + gf32::BM - 1) / gf32::BM, tiles_n = (N + gf32::BN - 1) / gf32::BN;
  uint32_t tm, tn;
  gemm::tile_coords<gf32::GROUP_M>(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const size_t co = static_cast<size_t>(blockIdx.y) * sc * OSZ;
  gemm_f32_tile_128<DT_OUT, B_TRANS, VEC, EPI>(
      A + blockIdx.y * sa, B + blockIdx.y * sb, static_cast<char*>(C) + co, M, N, K, tm, tn,
      up ? static_cast<const char*>(up) + co : nullptr);
}

// ============================================================================
// 64 x 64 tiles, for products whose 128 x 128 tiles would leave CUs idle.
//
// Bound: the fp32 matrix cores, once every SIMD has work.  999 x 4096 x 1000 is 64 tiles
// of 128 x 128 (a quarter of the chip, one wave per SIMD there) and 256 of 64 x 64.  Eight
// waves per workgroup, two per SIMD: wave (kh, wm, wn) computes 32 x 32 of the tile over
// half kh of every 64-deep K stage, and the two halves' sums are added through LDS at the
// end.  Two LDS stages; the next stage's values wait in registers while the current one
// computes.  A product with fewer tiles still is also split over K (grid z), f32 partials to
// a workspace that gemm_splitk_reduce adds in order.
//
// LDS holds A^T[k][m] and B[k][n], rows of 64 floats, column x of row k at
// x ^ 32 (k & 1) ^ 16 ((k >> 2) & 3): the two k rows of an MFMA operand read fall in
// opposite halves of the 64 banks, and so do (4 rows of 16 columns) the transposing
// writes, whose 16 lane groups then read 64 consecutive bytes of a matrix row each.
//
// Measured on MI355X: 999 x 4096 x 1000 522 -> 91 us (90 TFLOP/s), 1024^3 96 -> 27,
// 300 x 3000 x 500 397 -> 21, 64 x 4096 x 64 427 -> 10.  Counters at 999 x 4096 x 1000: MFMA
// busy 56%, 1.6 LDS instructions per MFMA, 14% of the LDS-active cycles in bank conflicts.
// ============================================================================
namespace gf32s {
constexpr int BM = 64, BN = 64, BK = 64;
constexpr int NT = 512;
using gf32::f32x16;
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// Values c .. c + 3 of a row of `cols`, zeros from `cols` on, without a branch on the lane
// and in two parts: fetch4 loads (a piece past the end reads the row's last four values),
// fix4 then makes the piece of what was loaded, so that only fix4 waits for the load.
// VEC: 16-byte aligned rows and cols % 4 == 0 (a piece is all inside or all outside).
template <bool VEC>
__device__ __forceinline__ f32x4 fetch4(const float* __restrict__ row, uint32_t c, uint32_t cols) {
  if constexpr (VEC) return *reinterpret_cast<const f32x4*>(row + min(c, cols - 4));
  if (cols >= 4) return *reinterpret_cast<const f32x4u*>(row + min(c, cols - 4));
  return f32x4{row[0], row[min(1u, cols - 1)], row[min(2u, cols - 1)], 0.0f};
}
template <bool VEC>
__device__ __forceinline__ f32x4 fix4(f32x4 w, uint32_t c, uint32_t cols) {
  if constexpr (VEC) return c < cols ? w : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // w holds values first .. first + 3 of the row
  const uint32_t first = cols >= 4 ? min(c, cols - 4) : 0u, sh = c - first;
  f32x4 v;
  v[0] = sh == 0 ? w[0] : sh == 1 ? w[1] : sh == 2 ? w[2] : sh == 3 ? w[3] : 0.0f;
  v[1] = sh == 0 ? w[1] : sh == 1 ? w[2] : sh == 2 ? w[3] : 0.0f;
  v[2] = sh == 0 ? w[2] : sh == 1 ? w[3] : 0.0f;
  v[3] = sh == 0 ? w[3] : 0.0f;
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = c + j < cols ? v[j] : 0.0f;
  return v;
}

struct alignas(16) Lds {
  float a[2][BK * BM];
  float b[2][BK * BN];
};
}  // namespace gf32s

// Tile (tm, tn) of C = A . B over k in [k0, k1); other arguments as gemm_f32_tile_128.
template <int DT_OUT, bool B_TRANS, bool VEC, int EPI>
__device__ __forceinline__ void gemm_f32_tile_64(const float* __restrict__ A,
                                                 const float* __restrict__ B,
                                                 void* __restrict__ C, uint32_t M, uint32_t N,
                                                 uint32_t K, uint32_t k0, uint32_t k1, uint32_t tm,
                                                 uint32_t tn, const void* __restrict__ up) {
  using namespace gf32s;
  __shared__ Lds s;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int kh = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
  const int h = lane >> 5, l32 = lane & 31;
  const uint32_t m0 = tm * BM, n0 = tn * BN;

  // Staging, two 16-byte pieces per thread and operand.  K-contiguous operands: piece i is
  // row tr, k 4 (tk + 8 i) .. +3; row-major B: k row bk + 32 i, columns 4 (lane % 16) .. +3.
  const int tr = 16 * (wave & 3) + (lane >> 2), tk = (lane & 3) + 4 * (wave >> 2);
  const int bk = 4 * wave + (lane >> 4), bn = 4 * (lane & 15);
  // Rows past M (N) read the last row (columns past N zeros): they reach only outputs that
  // are not stored.  Values past k1 are zero in both operands.
  const float* arow = A + static_cast<size_t>(min(m0 + tr, M - 1)) * K;
  const float* brow = B + static_cast<size_t>(min(n0 + tr, N - 1)) * K;   // B_TRANS
  f32x4 ra[2], rb[2];
  auto load = [&](uint32_t kb) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      ra[i] = fetch4<VEC>(arow, kb + 4 * (tk + 8 * i), k1);
      if constexpr (B_TRANS) rb[i] = fetch4<VEC>(brow, kb + 4 * (tk + 8 * i), k1);
      else
        rb[i] = fetch4<VEC>(B + static_cast<size_t>(min(kb + bk + 32 * i, k1 - 1)) * N, n0 + bn, N);
    }
  };
  const int tw = 256 * tk + (tr ^ (16 * (lane & 3)));   // row 4 tk, its column of tr
  auto put = [&](float* dst, const f32x4& v, int i) {
#pragma unroll
    for (int j = 0; j < 4; ++j) dst[(tw ^ (32 * (j & 1))) + 64 * j + 2048 * i] = v[j];
  };
  auto store = [&](int buf, uint32_t kb) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t kc = kb + 4 * (tk + 8 * i), kr = kb + bk + 32 * i;
      put(s.a[buf], fix4<VEC>(ra[i], kc, k1), i);
      if constexpr (B_TRANS) put(s.b[buf], fix4<VEC>(rb[i], kc, k1), i);
      else
        *reinterpret_cast<f32x4*>(
            &s.b[buf][64 * (bk + 32 * i) + (bn ^ (32 * (bk & 1)) ^ (16 * (wave & 3)))]) =
            kr < k1 ? fix4<VEC>(rb[i], n0 + bn, N) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  };

  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  // operand reads: k = 32 kh + 2 ks + h, (k >> 2) & 3 = (ks >> 1) & 3
  const int ko = 64 * (32 * kh + h);
  const int ao = ko + ((32 * wm + l32) ^ (32 * h)), bo = ko + ((32 * wn + l32) ^ (32 * h));

  const uint32_t nk = (k1 - k0 + BK - 1) / BK;
  load(k0);
  store(0, k0);
  if (nk > 1) load(k0 + BK);
  __syncthreads();
  for (uint32_t kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    // the next stage goes into the idle buffer, and the one after it is loaded, before this
    // stage's MFMAs: nothing but the barrier follows them
    if (kt + 1 < nk) store(cur ^ 1, k0 + (kt + 1) * BK);
    if (kt + 2 < nk) load(k0 + (kt + 2) * BK);
    const float* sa = s.a[cur];
    const float* sb = s.b[cur];
    // operands of two MFMAs (k rows 2 apart) per group, one group ahead of their use
    float fa[2], fb[2];
    auto frag = [&](int g) {
      const int x = 16 * (g & 3);
      fa[0] = sa[(ao ^ x) + 256 * g];
      fa[1] = sa[(ao ^ x) + 256 * g + 128];
      fb[0] = sb[(bo ^ x) + 256 * g];
      fb[1] = sb[(bo ^ x) + 256 * g + 128];
    };
    frag(0);
#pragma unroll
    for (int g = 0; g < BK / 8; ++g) {
      const float a0 = fa[0], a1 = fa[1], b0 = fb[0], b1 = fb[1];
      if (g + 1 < BK / 8) frag(g + 1);
      __builtin_amdgcn_sched_barrier(0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b0, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b1, acc, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
  }

  // add the two K halves: each wave hands its partner the 8 accumulators that the partner
  // stores (accumulator r: row 8 (r / 4) + 4 h + r % 4, column l32)
  float* x = s.a[0];
#pragma unroll
  for (int r = 0; r < 8; ++r) x[(8 * wave + r) * 64 + lane] = kh ? acc[r] : acc[8 + r];
  __syncthreads();
  const uint32_t col = n0 + 32 * wn + l32;
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const float v = (kh ? acc[8 + r] : acc[r]) + x[(8 * (wave ^ 4) + r) * 64 + lane];
    const uint32_t row = m0 + 32 * wm + 16 * kh + 8 * (r >> 2) + 4 * h + (r & 3);
    if (row < M && col < N)
      gemm::store_out<EPI, DT_OUT>(C, up, static_cast<size_t>(row) * N + col, v);
  }
}

// Library kernel: tiles in XCD-aware grouped order, batch = blockIdx.y (element strides sa,
// sb, sc), K slice = blockIdx.z: k [z ks, (z + 1) ks) to C + z M N (ks a multiple of 64; one
// slice: ks >= K).
template <int DT_OUT, bool B_TRANS, bool VEC, int EPI = 0>
__global__ void __launch_bounds__(gf32s::NT)
gemm_f32_64(const float* __restrict__ A, const float* __restrict__ B, void* __restrict__ C,
            uint32_t M, uint32_t N, uint32_t K, uint64_t sa, uint64_t sb, uint64_t sc,
            const void* __restrict__ up, uint32_t ks) {
  constexpr int OSZ = (DT_OUT == kF32) ? 4 : 2;
  uint32_t tm, tn;
  gemm::tile_coords<gf32::GROUP_M>(blockIdx.x, (M + gf32s::BM - 1) / gf32s::BM,
                                   (N + gf32s::BN - 1) / gf32s::BN, tm, tn);
  const size_t co = (static_cast<size_t>(blockIdx.y) * sc +
                     static_cast<size_t>(blockIdx.z) * M * N) * OSZ;
  const uint32_t k0 = blockIdx.z * ks;
  gemm_f32_tile_64<DT_OUT, B_TRANS, VEC, EPI>(
      A + blockIdx.y * sa, B + blockIdx.y * sb, static_cast<char*>(C) + co, M, N, K, k0,
      min(K - k0, ks) + k0, tm, tn, up ? static_cast<const char*>(up) + co : nullptr);
}

}  // namespace th
