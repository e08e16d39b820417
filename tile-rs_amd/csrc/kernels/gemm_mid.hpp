// 16-bit GEMM on tiles smaller than 256 x 256, for products that would leave CUs idle there:
// prompts of some hundred tokens, narrow outputs (K and V projections), and K not a
// multiple of 32.
//
// BM x BN tile (128 x 64 or 64 x 64) per four-wave workgroup, wave (w / 2, w % 2) a
// quarter of it in 16 x 16 blocks (v_mfma_f32_16x16x32).  K runs in 64-deep stages through a
// ring of NS LDS buffers filled by DMA, one barrier per stage: wait for the own share of
// stage i, barrier, refill the buffer of stage i - 1 with stage i + NS - 1, read and
// multiply.  Bound: the DMA stream and the barriers' latency; two workgroups share a CU
// (128 x 128 tiles, one per CU at four stages, were no faster anywhere between the two
// neighbours' ranges and are not kept).  Which tile when: plan_16bit in ops_gemm_mid.hip,
// with the figures.
//
// LDS: A (and B stored N x K) rows of 64 k, 128 bytes, 16-byte chunk c of row r at
// c ^ (r % 8); row-major B [64 k][BN], read as B^T with ds_read_b64_tr_b16, chunk c of k row
// r at c ^ sb(r), which keeps the rows and lane groups of one transposed read in distinct
// banks.  B is the MFMA's first operand, so a lane holds four consecutive columns of one row
// of C and stores them together.  Rows past M (columns past N) read the last ones and are
// not stored; past K both operands' fragments are zeroed.
//
// One 4096-deep tile per CU: 64 x 64 20.5 us, 128 x 64 30.5; two: 28 and 45; four: 54, 98.
#pragma once

#include "gemm.hpp"

namespace th {
namespace gmid {
constexpr int NT = 256;
constexpr int KB = 64;
template <int BM, int BN> constexpr int kStages = BM == 128 ? 3 : 4;   // two workgroups per CU

// Four values of a row of C from column col on; VEC: col % 4 == 0 columns are aligned.
template <int EPI, int DT_OUT>
__device__ __forceinline__ void store4(void* __restrict__ C, const void* __restrict__ up,
                                       size_t off, f32x4 v, uint32_t left, bool vec) {
  if (vec && left >= 4) {
    if constexpr (EPI == gemm::kEpiSiluMul) {
      float u[4];
      if constexpr (DT_OUT == kF32) {
        const f32x4 w = *reinterpret_cast<const f32x4*>(static_cast<const float*>(up) + off);
#pragma unroll
        for (int e = 0; e < 4; ++e) u[e] = w[e];
      } else {
        const u32x2 w = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(up) + off);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          u[e] = u16_to_f32<DT_OUT>(static_cast<uint16_t>(w[e >> 1] >> (16 * (e & 1))));
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = v[e] / (1.0f + expf(-v[e])) * u[e];
    }
    if constexpr (DT_OUT == kF32) {
      __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(static_cast<float*>(C) + off));
    } else {
      const u32x2 p = {pack2<DT_OUT>(v[0], v[1]), pack2<DT_OUT>(v[2], v[3])};
      __builtin_nontemporal_store(p, reinterpret_cast<u32x2*>(static_cast<uint16_t*>(C) + off));
    }
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (static_cast<uint32_t>(e) < left) gemm::store_out<EPI, DT_OUT>(C, up, off + e, v[e]);
}
}  // namespace gmid

// Tile (tm, tn) of C = epilogue(A . B) over k in [k0, k1) (k0 a multiple of 64); K % 8 == 0,
// row-major B N % 8 == 0, A and B 16-byte aligned.  vec: C (and UP) 16-byte aligned, N % 4
// == 0.
template <int DT, int DT_OUT, bool BT, int EPI, int BM, int BN>
__device__ __forceinline__ void gemm_mid_tile(const uint16_t* __restrict__ A,
                                              const uint16_t* __restrict__ B, void* __restrict__ C,
                                              uint32_t M, uint32_t N, uint32_t K, uint32_t k0,
                                              uint32_t k1, uint32_t tm, uint32_t tn,
                                              const void* __restrict__ up, bool vec) {
  using namespace gmid;
  constexpr int NS = kStages<BM, BN>;
  constexpr int SA = BM * 8, SB = BN * 8, ST = SA + SB;   // 16-byte slots per stage
  constexpr int NA = SA / NT, NB = SB / NT, ND = NA + NB;  // DMAs per wave and stage
  constexpr int MB = BM / 32, NBK = BN / 32;               // 16-wide blocks per wave
  u32x4* arena = lds::dma_lds_arena<NS * ST * 16>();
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int l16 = lane & 15, g = lane >> 4;
  const uint32_t m0 = tm * BM, n0 = tn * BN;

  // DMA j of this wave: 64 slots from 64 (NA wave + j) on
  const uint16_t* srcA[NA];
  const uint16_t* srcB[NB];
  int ka[NA], kb[NB];   // k of the lane's chunk (row-major B: k row) within a stage
#pragma unroll
  for (int j = 0; j < NA; ++j) {
    const int row = 8 * (NA * wave + j) + (lane >> 3);
    ka[j] = 8 * ((lane & 7) ^ (row & 7));
    srcA[j] = A + static_cast<size_t>(min(m0 + row, M - 1)) * K;
  }
  static_assert(BN == 64, "k rows of 128 bytes: sb and the transposed reads' offsets");
  auto sb = [](int r) { return 4 * ((r >> 1) & 1) ^ 2 * ((r >> 3) & 1); };
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    if constexpr (BT) {
      const int row = 8 * (NB * wave + j) + (lane >> 3);
      kb[j] = 8 * ((lane & 7) ^ (row & 7));
      srcB[j] = B + static_cast<size_t>(min(n0 + row, N - 1)) * K;
    } else {
      constexpr int CPR = BN / 8;   // chunks per k row
      const int slot = 64 * (NB * wave + j) + lane;
      kb[j] = slot / CPR;
      srcB[j] = B + min(n0 + 8 * ((slot % CPR) ^ sb(kb[j])), N - 8);
    }
  }
  const uint32_t n = (k1 - k0 + KB - 1) / KB;
  // stages past the last re-read it, so that the count in flight stays the same; chunks past
  // K read the last ones
  auto issue = [&](uint32_t i) {
    const uint32_t k = k0 + min(i, n - 1) * KB;
    u32x4* d = arena + (i % NS) * ST;
#pragma unroll
    for (int j = 0; j < NA; ++j)
      lds::dma16(srcA[j] + min(k + ka[j], K - 8), d + 64 * (NA * wave + j));
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const uint16_t* p = BT ? srcB[j] + min(k + kb[j], K - 8)
                             : srcB[j] + static_cast<size_t>(min(k + kb[j], K - 1)) * N;
      lds::dma16(p, d + SA + 64 * (NB * wave + j));
    }
  };

  f32x4 acc[NBK][MB];
#pragma unroll
  for (int j = 0; j < NBK; ++j)
#pragma unroll
    for (int i = 0; i < MB; ++i) acc[j][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  auto read_k = [&](const u32x4* s, int row, int h) {   // K-contiguous operand
    return s[row * 8 + ((4 * h + g) ^ (row & 7))];
  };
  // row-major B: byte offset in the stage of this lane's transposed reads of block j
  uint32_t tro[NBK];
  if constexpr (!BT) {
    const int kr = 8 * g + (l16 >> 2);
#pragma unroll
    for (int j = 0; j < NBK; ++j) {
      const int c = wn * (BN / 2) + 16 * j + 4 * (l16 & 3);
      tro[j] = kr * BN * 2 + (((c >> 3) ^ sb(kr)) << 4) + (c & 7) * 2;
    }
  }
  auto step = [&](uint32_t i, auto tail) {
    const u32x4* sa = arena + (i % NS) * ST;
    const u32x4* sbp = sa + SA;
    u32x4 a[2][MB], b[2][NBK];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int x = 0; x < MB; ++x) a[h][x] = read_k(sa, wm * (BM / 2) + 16 * x + l16, h);
      if constexpr (BT) {
#pragma unroll
        for (int x = 0; x < NBK; ++x) b[h][x] = read_k(sbp, wn * (BN / 2) + 16 * x + l16, h);
      }
    }
    if constexpr (!BT) {
      // inline asm: as builtins the compiler would order these after every DMA in flight
      const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds::lds_void*)(sbp)));
      u32x2 lo[2][NBK], hi[2][NBK];
#pragma unroll
      for (int x = 0; x < NBK; x += 2) {
        const uint32_t p0 = base + tro[x], p1 = base + tro[x + 1];
        asm volatile(
              "ds_read_b64_tr_b16 %0, %8\n"
              "ds_read_b64_tr_b16 %1, %8 offset:512\n"
              "ds_read_b64_tr_b16 %2, %9\n"
              "ds_read_b64_tr_b16 %3, %9 offset:512\n"
              "ds_read_b64_tr_b16 %4, %8 offset:4096\n"
              "ds_read_b64_tr_b16 %5, %8 offset:4608\n"
              "ds_read_b64_tr_b16 %6, %9 offset:4096\n"
              "ds_read_b64_tr_b16 %7, %9 offset:4608\n"
              "s_waitcnt lgkmcnt(0)"
              : "=&v"(lo[0][x]), "=&v"(hi[0][x]), "=&v"(lo[0][x + 1]), "=&v"(hi[0][x + 1]),
                "=&v"(lo[1][x]), "=&v"(hi[1][x]), "=&v"(lo[1][x + 1]), "=&v"(hi[1][x + 1])
              : "v"(p0), "v"(p1)
              : "memory");
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int x = 0; x < NBK; ++x)
          b[h][x] = u32x4{lo[h][x][0], lo[h][x][1], hi[h][x][0], hi[h][x][1]};
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if constexpr (decltype(tail)::value) {
        if (k0 + i * KB + 32 * h + 8 * g >= k1) {
#pragma unroll
          for (int x = 0; x < MB; ++x) a[h][x] = u32x4{0, 0, 0, 0};
#pragma unroll
          for (int x = 0; x < NBK; ++x) b[h][x] = u32x4{0, 0, 0, 0};
        }
      }
#pragma unroll
      for (int y = 0; y < NBK; ++y)
#pragma unroll
        for (int x = 0; x < MB; ++x) acc[y][x] = mfma16x16x32<DT>(b[h][y], a[h][x], acc[y][x]);
    }
  };

#pragma unroll
  for (int i = 0; i < NS - 1; ++i) issue(i);
  auto turn = [&](uint32_t i) {
    lds::wait_vm<(NS - 2) * ND>();
    lds::wait_lgkm0();   // the reads of stage i - 1
    lds::bar();
    issue(i + NS - 1);
  };
  const uint32_t whole = (k1 - k0) / KB;
  for (uint32_t i = 0; i < whole; ++i) {
    turn(i);
    step(i, std::false_type{});
  }
  if (whole < n) {
    turn(whole);
    step(whole, std::true_type{});
  }
  lds::wait_vm<0>();

  // D's column l % 16 is a row of C, its rows 4 (l / 16) + r four columns
#pragma unroll
  for (int x = 0; x < MB; ++x) {
    const uint32_t row = m0 + wm * (BM / 2) + 16 * x + l16;
    if (row >= M) continue;
#pragma unroll
    for (int y = 0; y < NBK; ++y) {
      const uint32_t col = n0 + wn * (BN / 2) + 16 * y + 4 * g;
      if (col < N)
        store4<EPI, DT_OUT>(C, up, static_cast<size_t>(row) * N + col, acc[y][x], N - col, vec);
    }
  }
}

// Grid: x = tiles in XCD-aware grouped order, y = batch (element strides sa, sb, sc), z = K
// slices of ks (a multiple of 64; more than one: DT_OUT f32, plain store, slice z to
// C + z M N).
template <int DT, int DT_OUT, bool BT, int EPI, int BM, int BN>
__global__ void __launch_bounds__(gmid::NT)
gemm_mid(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B, void* __restrict__ C,
         uint32_t M, uint32_t N, uint32_t K, uint64_t sa, uint64_t sb, uint64_t sc,
         const void* __restrict__ up, uint32_t ks, bool vec) {
  constexpr int OSZ = (DT_OUT == kF32) ? 4 : 2;
  uint32_t tm, tn;
  gemm::tile_coords(blockIdx.x, (M + BM - 1) / BM, (N + BN - 1) / BN, tm, tn);
  const size_t co = (static_cast<size_t>(blockIdx.y) * sc +
                     static_cast<size_t>(blockIdx.z) * M * N) * OSZ;
  const uint32_t k0 = blockIdx.z * ks;
  gemm_mid_tile<DT, DT_OUT, BT, EPI, BM, BN>(
      A + blockIdx.y * sa, B + blockIdx.y * sb, static_cast<char*>(C) + co, M, N, K, k0,
      k0 + min(K - k0, ks), tm, tn, up ? static_cast<const char*>(up) + co : nullptr, vec);
}

}  // namespace th
