// 16-bit products: the choice of tile and K split, and the kernels of tiles smaller than
// 256 x 256 (kernels/gemm_mid.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "kernels/gemm_mid.hpp"
#include "ops_gemm.hpp"

namespace th {
namespace ops {
namespace {

template <int DT, int DTO, int EPI, int BM, int BN>
int launch(const GemmArgs& g, void* c, uint32_t S, uint32_t ks) {
  const dim3 grid(((g.m + BM - 1) / BM) * ((g.n + BN - 1) / BN), g.batch, S), block(gmid::NT);
  constexpr uint64_t OSZ = DTO == kF32 ? 4 : 2;
  const bool vec = aligned16(c) && (!g.up || aligned16(g.up)) && g.n % 4 == 0 &&
                   (g.sc * OSZ) % 16 == 0;
  auto A = static_cast<const uint16_t*>(g.a);
  auto B = static_cast<const uint16_t*>(g.b);
  if (g.bt)
    hipLaunchKernelGGL((gemm_mid<DT, DTO, true, EPI, BM, BN>), grid, block, 0, g.s, A, B, c, g.m,
                       g.n, g.k, g.sa, g.sb, g.sc, g.up, ks, vec);
  else
    hipLaunchKernelGGL((gemm_mid<DT, DTO, false, EPI, BM, BN>), grid, block, 0, g.s, A, B, c, g.m,
                       g.n, g.k, g.sa, g.sb, g.sc, g.up, ks, vec);
  return launch_status("matmul (mid tiles) launch");
}

template <int DT, int DTO, int EPI>
int by_tile(const GemmArgs& g, void* c, const GemmPlan& p) {
  return p.tile == GemmPlan::k128x64 ? launch<DT, DTO, EPI, 128, 64>(g, c, p.slices, p.ks)
                                     : launch<DT, DTO, EPI, 64, 64>(g, c, p.slices, p.ks);
}

template <int DT, int EPI>
int go(const GemmArgs& g, th_dtype out, GemmPlan p) {
  void* ws = nullptr;
  ScratchHold hold;
  // No split without memory for the partials.  While a graph is recorded (nothing can be
  // allocated, and its replays could meet on the stream's scratch): only in place of a split
  // on 256 x 256 tiles, which shares that buffer too, and if it is large enough already.
  // (Row-major B 8 x 4096 x 1024 needs it: 16 workgroups unsplit.)
  const uint64_t bytes = static_cast<uint64_t>(p.slices) * g.m * g.n * sizeof(float);
  if (p.slices > 1 &&
      ((stream_capturing(g.s) && !(p.in_graph && th::stream_scratch_ready(g.s, bytes))) ||
       !th::try_stream_scratch(g.s, bytes, &ws, &hold))) {
    p.slices = 1;
    p.ks = g.k;
  }
  if (p.slices > 1) {
    GemmArgs part = g;
    part.up = nullptr;
    part.sc = 0;
    TH_TRY((by_tile<DT, kF32, gemm::kEpiStore>(part, ws, p)));
    return splitk_merge(g, static_cast<const float*>(ws), p.slices, out, EPI);
  }
  switch (out) {
    case TH_F32: return by_tile<DT, kF32, EPI>(g, g.c, p);
    case TH_F16: return by_tile<DT, kF16, EPI>(g, g.c, p);
    default: return by_tile<DT, kBF16, EPI>(g, g.c, p);
  }
}

}  // namespace

// Every form's time is estimated and the least taken.  Measured on MI355X for K = 4096 (us,
// linear in K, plus 3):
//   a round of 256 x 256 tiles: 66 on half the chip to 91 on all of it (B stored N x K and
//   over 64 MB: 100, 95 from the second round on), the LDS-DMA kernel 100 (105 N x K), the
//   register-staged one 155;
//   128 x 64 tiles max(30.5, 4 + 22.5 w), 64 x 64 tiles max(20.5, 5 + 13.5 w), w tiles per CU
//   (row-major B 1.12 times, rows off 128 bytes 1.3, B over 64 MB 1.08 to 1.4), no faster than
//   A and B come in at 3 TB/s (a line for these tiles alone: split 256 x 256 ones stream B
//   at 5.2 TB/s, row-major 8 x 14336 x 4096 22.4 against 23.9 at the best split of 64 x 64);
//   a K split adds 4 us and its f32 partials, written and read at 4 TB/s.
// E.g. (bf16, row-major, us, one box, against 256 x 256 tiles always, K split in as many equal
// slices of whole stages as give no CU two workgroups) 100 x 4096 x 4096 30 -> 18, 1000 x 4096 x
// 1024 53 -> 24, 4096 x 4096 x 1024 71 -> 47, 512 x 4096 x 4096 59 -> 36, 1000 x 4096 x 4096
// 71 -> 47, 2048 x 4096 x 4096 102 -> 65 (256 x 256, no split), 300 x 3752 x 2840 143 -> 22, 8 x
// 4096 x 1024 12.7 -> 7.9.
GemmPlan plan_16bit(const GemmArgs& g, const GemmForms& f) {
  const double cus = current_cu_count(), mn = static_cast<double>(g.m) * g.n;
  const double kk = g.k / 4096.0;
  const double in_bytes = 2.0 * g.k * (static_cast<double>(g.m) + g.n) * g.batch;
  const bool big_b = 2.0 * g.k * g.n > 64e6;
  auto merge_us = [&](uint32_t s) { return s > 1 ? 4.0 + s * mn * 8 / 4e6 : 0.0; };
  // 256 x 256
  const double t256 = std::ceil(g.m / 256.0) * std::ceil(g.n / 256.0);
  auto est256 = [&](uint32_t s) {
    const double w = t256 * g.batch * s / cus;
    const double per = s > 1 || !f.whole ? (!f.dma ? 155.0 : g.bt ? 105.0 : 100.0) * std::ceil(w)
                       : g.bt && big_b   ? (w <= 1.0 ? 100.0 : 95.0 * std::ceil(w))
                       : w <= 1.0        ? 66.0 + 50.0 * std::max(0.0, w - 0.5)
                                         : 91.0 * std::ceil(w);
    return 3.0 + per * kk / s + merge_us(s);
  };
  const bool in_graph = f.split > 1;
  GemmPlan best{GemmPlan::k256, 1, g.k, in_graph};
  double best_us = est256(1);
  if (f.split > 1 && est256(f.split) < best_us) {
    best = {GemmPlan::k256, f.split, g.k / f.split, in_graph};
    best_us = est256(f.split);
  }
  for (int tile : {GemmPlan::k128x64, GemmPlan::k64x64}) {
    const double bm = tile == GemmPlan::k128x64 ? 128.0 : 64.0;
    const double tiles = std::ceil(g.m / bm) * std::ceil(g.n / 64.0);
    const uint32_t most = g.batch == 1 && 2 * tiles <= cus ? std::min(32u, g.k / 256) : 1;
    for (uint32_t s = 1; s <= std::max(1u, most); ++s) {
      const uint32_t ks = s == 1 ? g.k : ((g.k + s - 1) / s + 63) / 64 * 64;
      if (s > 1 && (g.k + ks - 1) / ks != s) continue;
      const double w = tiles * g.batch * s / cus;
      double per = tile == GemmPlan::k128x64 ? std::max(30.5, 4.0 + 22.5 * w)
                                             : std::max(20.5, 5.0 + 13.5 * w);
      per *= (g.bt ? 1.0 : 1.12) * (g.k % 64 ? 1.3 : 1.0);
      if (big_b) per *= tile == GemmPlan::k128x64 ? (w > 1 ? 1.2 : 1.08) : g.bt ? 1.2 : 1.4;
      const double us = std::max(3.0 + per * ks / 4096.0, in_bytes / 3e6) + merge_us(s);
      if (us < best_us) {
        best = {tile, s, ks, in_graph};
        best_us = us;
      }
    }
  }
  return best;
}

int gemm_mid_tiles(const GemmArgs& g, th_dtype in, th_dtype out, int epi, const GemmPlan& p) {
  if (in == TH_F16)
    return epi == gemm::kEpiSiluMul ? go<kF16, gemm::kEpiSiluMul>(g, out, p)
                                    : go<kF16, gemm::kEpiStore>(g, out, p);
  return epi == gemm::kEpiSiluMul ? go<kBF16, gemm::kEpiSiluMul>(g, out, p)
                                  : go<kBF16, gemm::kEpiStore>(g, out, p);
}

}  // namespace ops
}  // namespace th
