// 16-bit products with few rows of A and B stored N x K (kernels/gemm_skinny.hpp).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "kernels/gemm_skinny.hpp"
#include "ops_gemm.hpp"

namespace th {
namespace ops {
namespace {

// 16-column blocks per workgroup: as many as leave four workgroups for five CUs (A is then
// re-read less often).
uint32_t col_blocks(const GemmArgs& g) {
  uint32_t nf = 1;
  while (nf < 4 && 5ull * ((g.n + 32 * nf - 1) / (32 * nf)) * g.batch >= 4ull * current_cu_count())
    nf *= 2;
  return nf;
}

template <int DT, int DTO, int EPI>
int launch(const GemmArgs& g) {
  const uint32_t nf = col_blocks(g);
  const dim3 grid((g.n + 16 * nf - 1) / (16 * nf), g.batch), block(gskinny::NT);
  auto go = [&](auto xr, auto f) {
    hipLaunchKernelGGL((gemm_skinny<DT, DTO, EPI, xr.value, f.value>), grid, block, 0, g.s,
                       static_cast<const uint16_t*>(g.a), static_cast<const uint16_t*>(g.b), g.c,
                       g.m, g.n, g.k, g.sa, g.sb, g.sc, g.up);
  };
  auto by_nf = [&](auto xr) {
    if (nf == 1) go(xr, std::integral_constant<int, 1>{});
    else if (nf == 2) go(xr, std::integral_constant<int, 2>{});
    else go(xr, std::integral_constant<int, 4>{});
  };
  if (g.m <= 8) by_nf(std::integral_constant<int, 8>{});
  else if (g.m <= 16) by_nf(std::integral_constant<int, 16>{});
  else if (g.m <= 32) by_nf(std::integral_constant<int, 32>{});
  else by_nf(std::integral_constant<int, 64>{});
  return launch_status("matmul (few rows) launch");
}

template <int DT, int EPI>
int by_out(const GemmArgs& g, th_dtype out) {
  switch (out) {
    case TH_F32: return launch<DT, kF32, EPI>(g);
    case TH_F16: return launch<DT, kF16, EPI>(g);
    default: return launch<DT, kBF16, EPI>(g);
  }
}

}  // namespace

// The line is where re-reading A costs more than the split-K kernel's partials and merge:
// re-reads of 134 MB (M 64, 4096 x 4096) 10.5 us here against 15.2, 117 MB (M 64, N 14336,
// K 4096) 28.9 against 37.5, but 235 MB (M 32, N 4096, K 14336) 30.7 against 29.6.
bool few_rows_fit(const GemmArgs& g) {
  if (!g.bt || g.m > gskinny::kMaxM) return false;
  const uint64_t groups = (g.n + 16 * col_blocks(g) - 1) / (16 * col_blocks(g));
  return groups * g.batch * g.m * g.k * 2 <= 180ull << 20;
}

int gemm_few_rows(const GemmArgs& g, th_dtype in, th_dtype out, int epi) {
  if (in == TH_F16)
    return epi == gemm::kEpiSiluMul ? by_out<kF16, gemm::kEpiSiluMul>(g, out)
                                    : by_out<kF16, gemm::kEpiStore>(g, out);
  return epi == gemm::kEpiSiluMul ? by_out<kBF16, gemm::kEpiSiluMul>(g, out)
                                  : by_out<kBF16, gemm::kEpiStore>(g, out);
}

}  // namespace ops
}  // namespace th
