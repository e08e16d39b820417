// GEMM entry points of the C ABI (include/tilers_hip.h, section 2): th_matmul and
// th_matmul_silu_mul, and their kernels for 16-bit operands (f32: ops_gemm_f32.hip).
// Shapes and pointers are checked on the host, the hand-written gfx950 kernel for the
// shape is picked and enqueued on the caller's stream; there is no CPU fallback.  (Its own translation unit: the GEMM instantiations compile in
// parallel with the rest of the library.)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>

#include "kernels/common.hpp"
#include "kernels/gemm.hpp"
#include "kernels/gemm_asm.hpp"
#include "ops_gemm.hpp"

using th::fail;
using namespace th::ops;

namespace {

// ---- matmul -------------------------------------------------------------------

// The LDS-DMA pipeline takes every shape with K % 32 == 0 that stays on 256 x 256 tiles, unless
// TILERS_HIP_GEMM_DMA=0 (a debugging switch: the register-staged kernel then
// runs them too).
bool gemm_dma() {
  static const bool v = [] {
    const char* e = std::getenv("TILERS_HIP_GEMM_DMA");
    return !(e && std::atoi(e) == 0);
  }();
  return v;
}

// Whole-tile shapes (B row-major or stored N x K) run on the generated-assembly kernel
// (gemm_asm.hpp) unless TILERS_HIP_GEMM_ASM=0 (a debugging switch: the LDS-DMA
// kernel, which gives the same bits for the plain store, then runs them).  Read on
// every call (a getenv, next to a kernel launch), so a process can compare the two.
bool gemm_asm() {
  const char* e = std::getenv("TILERS_HIP_GEMM_ASM");
  return !(e && std::atoi(e) == 0);
}

// Split-K for shapes with too few 256 x 256 tiles to fill the chip (small M:
// decode-time projections).  S slices of K (each a multiple of 32, at least 256
// deep, S a divisor of K / 32) run as the batch dimension of the DMA kernel,
// writing f32 partials to a per-stream workspace; gemm_splitk_reduce adds them
// and applies the epilogue.  Only for batch 1.  Returns 1 for no split.
uint32_t splitk_slices(const GemmArgs& g, uint32_t tiles) {
  const uint32_t cus = current_cu_count();
  if (g.batch != 1 || 2u * tiles > cus || g.k < 512) return 1;
  const uint32_t units = g.k / th::gemm::DBK;             // K in 32-deep steps
  const uint32_t cap = std::min<uint32_t>({cus / tiles, g.k / 256u, 32u});
  uint32_t best = 1;
  for (uint32_t s = 2; s <= cap; ++s)
    if (units % s == 0) best = s;
  return best;
}

template <int DT, int DTO, int EPI, bool BT>
int gemm_splitk(const GemmArgs& g, uint32_t tiles, uint32_t S) {
  const uint32_t ks = g.k / S;
  const uint64_t mn = static_cast<uint64_t>(g.m) * g.n;
  void* wv = nullptr;
  th::ScratchHold hold;
  TH_TRY(th::stream_scratch(g.s, S * mn * sizeof(float), &wv, &hold));
  auto* W = static_cast<float*>(wv);
  auto go = [&](auto mi) {
    constexpr int MI = decltype(mi)::value;
    hipLaunchKernelGGL((th::gemm_dma_256<DT, th::kF32, BT, th::gemm::DBK, th::gemm::NSTAGE,
                                         th::gemm::DWAVES, th::gemm::kEpiStore, MI>),
                       dim3(tiles, S), dim3(64 * th::gemm::DWAVES), 0, g.s,
                       static_cast<const uint16_t*>(g.a), static_cast<const uint16_t*>(g.b),
                       static_cast<void*>(W), g.m, g.n, ks, static_cast<uint64_t>(ks),
                       BT ? static_cast<uint64_t>(ks) : static_cast<uint64_t>(ks) * g.n, mn,
                       static_cast<const void*>(nullptr), g.k);
  };
  // rows past M are padding: compute only the 32-row blocks that hold real rows
  if (g.m <= 32) go(std::integral_constant<int, 1>{});
  else if (g.m <= 64) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 4>{});
  TH_TRY(launch_status("matmul (split-K) launch"));
  return splitk_merge(g, W, S,
                      DTO == th::kF32 ? TH_F32 : DTO == th::kF16 ? TH_F16 : TH_BF16, EPI);
}

// Whether the LDS-DMA pipeline takes the product (its SiLU*Mul epilogue writes C and reads UP
// in 16-byte pieces).
bool dma_fits(const GemmArgs& g, int epi, uint64_t osz) {
  return gemm_dma() && g.k % th::gemm::DBK == 0 &&
         (epi != th::gemm::kEpiSiluMul ||
          (aligned16(g.c) && aligned16(g.up) && (g.sc * osz) % 16 == 0 && g.n % 8 == 0));
}

// Whether UP and C share memory.
bool overlap(const GemmArgs& g, uint64_t osz) {
  const uint64_t n = ((g.batch - 1) * g.sc + static_cast<uint64_t>(g.m) * g.n) * osz;
  const auto c = reinterpret_cast<uintptr_t>(g.c), up = reinterpret_cast<uintptr_t>(g.up);
  return c < up + n && up < c + n;
}

template <int DT, int DTO, int EPI, bool BT>
int gemm_mfma_go(const GemmArgs& g, dim3 grid) {
  auto A = static_cast<const uint16_t*>(g.a);
  auto B = static_cast<const uint16_t*>(g.b);
  constexpr uint64_t OSZ = (DTO == th::kF32) ? 4 : 2;
  if (dma_fits(g, EPI, OSZ)) {
    if (g.slices > 1) return gemm_splitk<DT, DTO, EPI, BT>(g, grid.x, g.slices);
    // Ragged M or N included (SiLU*Mul, 3000 x 4096 x 14336 f16: 288 us here, 352 us on the
    // LDS-DMA kernel)
    const bool fits = th::gasm::fits(g.m, g.n, g.k, static_cast<int>(OSZ)) && gemm_asm();
    if constexpr (EPI == th::gemm::kEpiStore) {
      if (fits) {
        hipLaunchKernelGGL((th::gemm_asm_256<DT, DTO, BT>), grid, dim3(th::gasm::NT), 0, g.s, A,
                           B, g.c, g.m, g.n, g.k, g.sa, g.sb, g.sc, nullptr);
        return launch_status("matmul (MFMA asm) launch");
      }
    } else if constexpr (DTO != th::kF32) {
      // SiLU*Mul with 16-bit C (UP staged through LDS: 16-byte aligned, checked above).
      // Tiles that share rows or columns read UP where the other may have written C, so
      // in place only whole tiles run it.
      if (fits && ((g.m % 256 == 0 && g.n % 256 == 0) || !overlap(g, OSZ))) {
        hipLaunchKernelGGL((th::gemm_asm_256<DT, DTO, BT, true>), grid, dim3(th::gasm::NT), 0, g.s,
                           A, B, g.c, g.m, g.n, g.k, g.sa, g.sb, g.sc, g.up);
        return launch_status("matmul silu*mul (MFMA asm) launch");
      }
    }
    hipLaunchKernelGGL((th::gemm_dma_256<DT, DTO, BT, th::gemm::DBK, th::gemm::NSTAGE,
                                         th::gemm::DWAVES, EPI>),
                       grid, dim3(64 * th::gemm::DWAVES), 0, g.s, A, B, g.c, g.m, g.n, g.k, g.sa,
                       g.sb, g.sc, g.up, 0u);
  } else if (g.m % th::gemm::BM == 0 && g.n % th::gemm::BN == 0 && g.k % th::gemm::BK == 0) {
    hipLaunchKernelGGL((th::gemm_mfma_256<DT, DTO, BT, 2, 2, true, EPI>), grid, dim3(256), 0, g.s,
                       A, B, g.c, g.m, g.n, g.k, g.sa, g.sb, g.sc, g.up);
  } else {
    hipLaunchKernelGGL((th::gemm_mfma_256<DT, DTO, BT, 2, 2, false, EPI>), grid, dim3(256), 0, g.s,
                       A, B, g.c, g.m, g.n, g.k, g.sa, g.sb, g.sc, g.up);
  }
  return launch_status("matmul (MFMA) launch");
}

template <int DT, int DTO, int EPI>
int gemm_launch(const GemmArgs& g, bool mfma) {
  if (mfma) {
    const dim3 grid(((g.m + 255) / 256) * ((g.n + 255) / 256), g.batch);
    return g.bt ? gemm_mfma_go<DT, DTO, EPI, true>(g, grid)
                : gemm_mfma_go<DT, DTO, EPI, false>(g, grid);
  }
  const dim3 grid(((g.m + 63) / 64) * ((g.n + 63) / 64), g.batch), block(256);
  if (g.bt)
    hipLaunchKernelGGL((th::gemm_fma_64<DT, DTO, true, EPI>), grid, block, 0, g.s, g.a, g.b, g.c,
                       g.m, g.n, g.k, g.sa, g.sb, g.sc, g.up);
  else
    hipLaunchKernelGGL((th::gemm_fma_64<DT, DTO, false, EPI>), grid, block, 0, g.s, g.a, g.b, g.c,
                       g.m, g.n, g.k, g.sa, g.sb, g.sc, g.up);
  return launch_status("matmul (FMA) launch");
}

template <int EPI>
int gemm_dispatch(const GemmArgs& g, th_dtype in, th_dtype out) {
  if (in == TH_F32) return gemm_f32(g, out, EPI);
  // the 16-bit MFMA paths need K % 8 == 0, row-major B N % 8 == 0 and 16-byte aligned
  // operands and strides
  const bool mfma = (g.k % 8 == 0) && (g.bt || g.n % 8 == 0) && aligned16(g.a) &&
                    aligned16(g.b) && (g.sa % 8 == 0) && (g.sb % 8 == 0);
  if (mfma && few_rows_fit(g)) return gemm_few_rows(g, in, out, EPI);
  GemmArgs h = g;
  if (mfma) {
    const uint64_t osz = dtype_size(out);
    GemmForms f{false, dma_fits(g, EPI, osz), 1};
    if (f.dma) {
      // (whatever TILERS_HIP_GEMM_ASM says: it swaps kernels on the same tiles and K split)
      f.whole = th::gasm::fits(g.m, g.n, g.k, static_cast<int>(osz)) &&
                (EPI == th::gemm::kEpiStore || out != TH_F32);
      f.split = splitk_slices(g, ((g.m + 255) / 256) * ((g.n + 255) / 256));
    }
    const GemmPlan plan = plan_16bit(g, f);
    if (plan.tile != GemmPlan::k256) return gemm_mid_tiles(g, in, out, EPI, plan);
    h.slices = plan.slices;
  }
  auto by_out = [&](auto dt) {
    constexpr int DT = decltype(dt)::value;
    switch (out) {
      case TH_F32: return gemm_launch<DT, th::kF32, EPI>(h, mfma);
      case TH_F16: return gemm_launch<DT, th::kF16, EPI>(h, mfma);
      default: return gemm_launch<DT, th::kBF16, EPI>(h, mfma);
    }
  };
  if (in == TH_F16) return by_out(std::integral_constant<int, th::kF16>{});
  return by_out(std::integral_constant<int, th::kBF16>{});
}

}  // namespace

namespace th {
namespace ops {

int splitk_merge(const GemmArgs& g, const float* W, uint32_t S, th_dtype out, int epi) {
  const uint64_t mn = static_cast<uint64_t>(g.m) * g.n;
  const uint32_t blocks = static_cast<uint32_t>(
      std::min<uint64_t>((mn + 255) / 256, 4ull * current_cu_count()));
  auto go = [&](auto dto, auto e) {
    hipLaunchKernelGGL((th::gemm_splitk_reduce<dto.value, e.value>), dim3(blocks), dim3(256), 0,
                       g.s, W, g.c, g.up, mn, S);
  };
  auto by_epi = [&](auto dto) {
    if (epi == th::gemm::kEpiSiluMul) go(dto, std::integral_constant<int, th::gemm::kEpiSiluMul>{});
    else go(dto, std::integral_constant<int, th::gemm::kEpiStore>{});
  };
  switch (out) {
    case TH_F32: by_epi(std::integral_constant<int, th::kF32>{}); break;
    case TH_F16: by_epi(std::integral_constant<int, th::kF16>{}); break;
    default: by_epi(std::integral_constant<int, th::kBF16>{}); break;
  }
  return launch_status("matmul (split-K merge) launch");
}

}  // namespace ops
}  // namespace th

extern "C" {

int th_matmul(const void* a, const void* b, void* c, uint32_t m, uint32_t k, uint32_t n,
              th_dtype in_dtype, th_dtype out_dtype, int b_transposed, uint32_t batch, uint64_t sa,
              uint64_t sb, uint64_t sc, th_stream s) {
  if (!valid_dtype(in_dtype) || !valid_dtype(out_dtype))
    return fail(TH_KERNEL_ERROR, "matmul: unknown dtype");
  if (m == 0 || n == 0 || batch == 0) return TH_OK;
  if (!a || !b || !c) return fail(TH_KERNEL_ERROR, "matmul: null pointer");
  if (batch > 65535) return fail(TH_KERNEL_ERROR, "matmul: batch > 65535");
  const bool bt = b_transposed != 0;
  if (sa == 0) sa = static_cast<uint64_t>(m) * k;
  if (sb == 0) sb = static_cast<uint64_t>(k) * n;
  if (sc == 0) sc = static_cast<uint64_t>(m) * n;
  if (k == 0) {
    // empty contraction: C = 0 (linalg.fill 0 with nothing accumulated)
    const size_t esz = dtype_size(out_dtype);
    for (uint32_t i = 0; i < batch; ++i)
      TH_TRY(th::check_hip(hipMemsetAsync(static_cast<char*>(c) + i * sc * esz, 0,
                                          static_cast<size_t>(m) * n * esz, as_stream(s)),
                           "hipMemsetAsync", TH_MEMORY_ERROR));
    return TH_OK;
  }
  const GemmArgs g{a, b, c, nullptr, m, k, n, bt, batch, sa, sb, sc, as_stream(s)};
  return gemm_dispatch<th::gemm::kEpiStore>(g, in_dtype, out_dtype);
}

int th_matmul_silu_mul(const void* a, const void* b, const void* up, void* c, uint32_t m,
                       uint32_t k, uint32_t n, th_dtype in_dtype, th_dtype out_dtype,
                       int b_transposed, uint32_t batch, uint64_t sa, uint64_t sb, uint64_t sc,
                       th_stream s) {
  if (!valid_dtype(in_dtype) || !valid_dtype(out_dtype))
    return fail(TH_KERNEL_ERROR, "matmul_silu_mul: unknown dtype");
  if (m == 0 || n == 0 || batch == 0) return TH_OK;
  if (!a || !b || !c || !up) return fail(TH_KERNEL_ERROR, "matmul_silu_mul: null pointer");
  if (batch > 65535) return fail(TH_KERNEL_ERROR, "matmul_silu_mul: batch > 65535");
  const bool bt = b_transposed != 0;
  if (sa == 0) sa = static_cast<uint64_t>(m) * k;
  if (sb == 0) sb = static_cast<uint64_t>(k) * n;
  if (sc == 0) sc = static_cast<uint64_t>(m) * n;
  if (k == 0) {
    // silu(0) * up = 0 everywhere
    const size_t esz = dtype_size(out_dtype);
    for (uint32_t i = 0; i < batch; ++i)
      TH_TRY(th::check_hip(hipMemsetAsync(static_cast<char*>(c) + i * sc * esz, 0,
                                          static_cast<size_t>(m) * n * esz, as_stream(s)),
                           "hipMemsetAsync", TH_MEMORY_ERROR));
    return TH_OK;
  }
  const GemmArgs g{a, b, c, up, m, k, n, bt, batch, sa, sb, sc, as_stream(s)};
  return gemm_dispatch<th::gemm::kEpiSiluMul>(g, in_dtype, out_dtype);
}

}  // extern "C"
