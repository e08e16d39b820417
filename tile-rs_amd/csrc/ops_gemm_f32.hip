// th_matmul / th_matmul_silu_mul on f32 operands: the fp32 MFMA kernels of
// kernels/gemm_f32.hpp and the choice of tile and K split.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "kernels/gemm_f32.hpp"
#include "ops_gemm.hpp"

namespace th {
namespace ops {
namespace {

// K slices of a product of `tiles` 64 x 64 tiles, each `ks` deep (a multiple of 64), and the
// workspace for their partials; 1 (and ks = K) for no split.  A CU works through its
// ceil(tiles S / CUs) workgroups at about 25 ns per k each (measured: 999 x 4096 x 1000,
// one per CU, 102 us), and a split adds the merge: about 4 us and the partials' bytes, written
// and read at about 4 TB/s.  The S with the least sum is taken.  No split while a graph is
// recorded (its replays could meet on the stream's scratch) or without memory for it.
uint32_t f32_slices(const GemmArgs& g, uint32_t tiles, uint32_t* ks, void** ws,
                    ScratchHold* hold) {
  *ks = g.k;
  if (g.batch != 1) return 1;
  const double cus = current_cu_count(), mn = static_cast<double>(g.m) * g.n;
  uint32_t best = 1;
  double best_ns = 0;
  for (uint32_t s = 1; s <= std::min(32u, std::max(1u, g.k / 128)); ++s) {
    const uint32_t d = ((g.k + s - 1) / s + 63) / 64 * 64, n = (g.k + d - 1) / d;
    if (n != s) continue;
    const double rounds = std::ceil(tiles * static_cast<double>(s) / cus);
    const double ns = 25.0 * rounds * std::min(d, g.k) + (s > 1 ? 4000.0 + s * mn * 8 / 4000.0 : 0.0);
    if (s == 1 || ns < best_ns) {
      best = s;
      best_ns = ns;
    }
  }
  if (best == 1 || stream_capturing(g.s) ||
      !th::try_stream_scratch(g.s, best * static_cast<uint64_t>(g.m) * g.n * sizeof(float), ws,
                              hold))
    return 1;
  *ks = ((g.k + best - 1) / best + 63) / 64 * 64;
  return best;
}

template <int DTO, int EPI>
int go(const GemmArgs& g, th_dtype out) {
  // 16-byte loads when every row start is 16-byte aligned
  const bool vec = aligned16(g.a) && aligned16(g.b) && g.k % 4 == 0 && (g.bt || g.n % 4 == 0) &&
                   g.sa % 4 == 0 && g.sb % 4 == 0;
  auto by_form = [&](auto launch) {
    if (g.bt) {
      if (vec) launch(std::true_type{}, std::true_type{});
      else launch(std::true_type{}, std::false_type{});
    } else {
      if (vec) launch(std::false_type{}, std::true_type{});
      else launch(std::false_type{}, std::false_type{});
    }
  };
  auto A = static_cast<const float*>(g.a);
  auto B = static_cast<const float*>(g.b);
  const uint64_t tiles = static_cast<uint64_t>((g.m + gf32::BM - 1) / gf32::BM) *
                         ((g.n + gf32::BN - 1) / gf32::BN);
  // 128 x 128 tiles run four to a CU, so they pay from four per CU on (4096 x 2048 x 4096,
  // 1024 tiles: 575 us against 632 us in 64 x 64; 3500 x 1000 x 3500, 784: 299 against 252;
  // 2048^3, 256: 189 against 162; 999 x 4096 x 1000, 64: 521 against 101; 64 x 4096 x 64:
  // 427 against 10 with K split)
  if (tiles * g.batch < 4ull * current_cu_count()) {
    const uint32_t t64 = ((g.m + gf32s::BM - 1) / gf32s::BM) * ((g.n + gf32s::BN - 1) / gf32s::BN);
    void* ws = nullptr;
    uint32_t ks = 0;
    ScratchHold hold;
    const uint32_t S = f32_slices(g, t64, &ks, &ws, &hold);
    const dim3 grid(t64, g.batch, S), block(gf32s::NT);
    if (S > 1) {
      by_form([&](auto bt, auto v) {
        hipLaunchKernelGGL((gemm_f32_64<kF32, bt.value, v.value>), grid, block, 0, g.s, A, B, ws,
                           g.m, g.n, g.k, 0, 0, 0, nullptr, ks);
      });
      TH_TRY(launch_status("matmul (fp32 MFMA, split K) launch"));
      return splitk_merge(g, static_cast<const float*>(ws), S, out, EPI);
    }
    by_form([&](auto bt, auto v) {
      hipLaunchKernelGGL((gemm_f32_64<DTO, bt.value, v.value, EPI>), grid, block, 0, g.s, A, B,
                         g.c, g.m, g.n, g.k, g.sa, g.sb, g.sc, g.up, ks);
    });
    return launch_status("matmul (fp32 MFMA) launch");
  }
  const dim3 grid(static_cast<uint32_t>(tiles), g.batch), block(gf32::NT);
  by_form([&](auto bt, auto v) {
    hipLaunchKernelGGL((gemm_f32_mfma<DTO, bt.value, v.value, EPI>), grid, block, 0, g.s, A, B,
                       g.c, g.m, g.n, g.k, g.sa, g.sb, g.sc, g.up);
  });
  return launch_status("matmul (fp32 MFMA) launch");
}

template <int EPI>
int by_out(const GemmArgs& g, th_dtype out) {
  switch (out) {
    case TH_F32: return go<kF32, EPI>(g, out);
    case TH_F16: return go<kF16, EPI>(g, out);
    default: return go<kBF16, EPI>(g, out);
  }
}

}  // namespace

int gemm_f32(const GemmArgs& g, th_dtype out, int epi) {
  return epi == gemm::kEpiSiluMul ? by_out<gemm::kEpiSiluMul>(g, out)
                                  : by_out<gemm::kEpiStore>(g, out);
}

}  // namespace ops
}  // namespace th
