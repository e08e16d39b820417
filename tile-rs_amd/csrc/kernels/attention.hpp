// Attention kernels: GQA decode (split-KV, MFMA scores), a general online-softmax
// kernel for every other shape/dtype, and the constants and work order of the
// causal GQA prefill (its 16-bit kernel is in prefill_asm.hpp; f32 single-head
// attention and f32 prefill are in attention_f32.hpp).
//
// Semantics (reference):
//   prefill  __tile_attention_prefill_f32  crates/tile_std/src/tile.rs:2136, :3064;
//            Metal template mlir_to_msl.rs:10928-11009, host params :1851-1859.
//            query qi of head h sits at absolute position start_pos + qi and sees
//            KV positions pos <= start_pos + qi of kv_head = h / (NH / NKV);
//            scale = rsqrt(D).
//   decode   __tile_attention_decode_f32   tile.rs:2124, :3011; mlir_to_msl.rs:
//            10747-10816, host params :1816-1823: one query per head, positions
//            [0, seq_len), same GQA map and scale.
//   single   __tile_attention_f32          tile.rs:221, :2401; linalg
//            decomposition mlir_to_linalg.rs:1781-1902 (non-causal, one head,
//            scale 1/sqrt(D) computed in f64 then rounded to f32).
// Layouts in HBM: Q, O = [B][S][NH][D]; K, V = [B][NKV][max_seq][D] (the Metal
// templates' per-batch layout, stacked over the batch).  The Metal templates cap
// the KV length at 256; these kernels have no cap.
#pragma once

#include "common.hpp"
#include "gemm.hpp"

namespace th {

// ============================================================================
// Prefill: flash attention forward, causal, GQA, head_dim 128.
//
// Workgroup = 8 waves = 256 query rows of one (batch, head); wave w owns rows
// [32w, 32w+32).  KV is consumed 64 positions at a time.  Per wave and KV block:
//   S^T (64 kv x 32 q)  = K . Q^T          2x8 v_mfma_f32_32x32x16, Q^T in registers
//   online softmax on S^T columns: lane l owns query l%32; its partner lane l^32
//   holds the other half of that column, so row statistics need one exchange.
//   O^T (128 d x 32 q) += V^T . P^T        4x4 MFMAs; P^T is the S^T accumulator
//   converted to 16-bit in place: accumulator j of lane l (half g = l/32) is KV
//   row 8*(j/4) + 4g + j%4, and the V^T operand is read in the same KV order, so
//   the B operand needs no data movement.
// The kernel is pfa::attn_prefill_asm (prefill_asm.hpp); its main loop is gfx950
// assembly generated by gen_prefill.py.  The constants and the work order below
// are shared with it and with the emitted prefill.
// ============================================================================
namespace fa {
constexpr int D = 128;
constexpr int BQ = 256;   // query rows per workgroup
constexpr int NT = 512;   // threads per workgroup (8 waves)
// A KV block whose probability mass exceeds 1/ratio of the query's running sum
// gets its P residual as well (bf16 keeps 8 significant bits, f16 keeps 11).
template <int DT> constexpr float kSplitRatio = (DT == kBF16) ? 16.0f : 2.0f;
}  // namespace fa

// Map a work index to (bh, qb).  The unit of K/V sharing is a (batch, kv head) pair
// with its G = nh / nkv query heads.  When the unit count allows, units are dealt to
// the 8 XCDs (work index w runs on XCD w % 8), and each XCD works through its units
// a few at a time: a group of about four query heads, and within the group heavy
// (late) query blocks first, the group's heads interleaved.  The query blocks of a
// group then stream the same K/V blocks close together in time, so most K/V loads
// hit that XCD's L2 (config 4, measured on MI355X: 594-596 us against 615-617 us
// when each XCD runs all of its 16 heads at once).
__device__ __forceinline__ void prefill_work(uint32_t w, uint32_t batch, uint32_t nh,
                                             uint32_t nkv, uint32_t nqb, uint32_t& bh,
                                             uint32_t& qb) {
  const uint32_t g = nh / nkv, units = batch * nkv;
  if (units % 8 == 0) {
    const uint32_t per = units / 8;
    uint32_t gu = g >= 4 ? 1 : 4 / g;   // units per group
    while (per % gu != 0) gu >>= 1;
    const uint32_t heads = gu * g;        // query heads per group
    const uint32_t xcd = w % 8, r = w / 8;
    const uint32_t grp = r / (heads * nqb), in = r % (heads * nqb);
    const uint32_t hs = in % heads;
    const uint32_t u = xcd + 8 * (grp * gu + hs / g);
    bh = (u / nkv) * nh + (u % nkv) * g + hs % g;
    qb = nqb - 1 - in / heads;
  } else {
    const uint32_t nbh = batch * nh;
    bh = w % nbh;
    qb = nqb - 1 - w / nbh;
  }
}

// ============================================================================
// Decode: one query token per head, GQA group G = NH/NKV query heads share each
// K/V load.  Grid = B * NKV * n_split workgroups of 256 threads; each walks a
// run of consecutive 512-position chunks of one (batch, kv_head), per chunk:
//   A  scores S^T (16 kv x 16 q, G real columns) with v_mfma_f32_16x16x32 (f32:
//      v_mfma_f32_16x16x4_f32), K fragments read straight from HBM (each lane 4, f32
//      8, x 16 B of one K row),
//   B  per-query max / exp / sum over the chunk (in LDS), merged into the
//      running (m, l) of the workgroup's run,
//   C  P.V on the vector ALUs in f32: each lane owns 8 d-values of every 4th row (f32:
//      4 of every 2nd).
// With one split the workgroup writes O itself; otherwise each run's partial
// (m, l, O) goes to a workspace and attn_decode_combine merges them.
// K and V are read exactly once, with nontemporal loads (measured on MI355X:
// ~8% more sustained bandwidth than cached loads for this stream).  f32, 8 sequences
// of 3000 positions, 32 heads over 8, D 128: 45.7 us (4.3 TB/s) against 536 us on the
// general kernel.
// ============================================================================
namespace dec {
constexpr int D = 128;
constexpr int CHUNK = 512;
constexpr int NT = 256;
constexpr int CT = 512;  // threads of the combine block
// decode_tile's LDS (scores, per-wave O, row statistics) sized for up to AG query
// heads and head dim AD: one variable for every instantiation that names the same
// (AG, AD), so a kernel that picks G and HD at run time can hold the largest layout
// rather than the sum of all of them.
template <int AG, int AD>
__device__ __forceinline__ float* lds_arena() {
  __shared__ __align__(16) float a[AG * (CHUNK + 16) + 4 * AG * AD + 3 * AG];
  return a;
}
}  // namespace dec

template <int DT> struct elem { using type = uint16_t; };
template <> struct elem<kF32> { using type = float; };
template <int DT> using elem_t = typename elem<DT>::type;

// One work item: chunks [c_begin, c_end) of (batch, kv_head) `bk` = b*NKV + kvh.
// With `ws` non-null the chunk range's partial (m, l, O) goes to
// ws[((bk*G + q)*n_split + split)*(D+2)]; otherwise O = acc / l is written to
// `O` directly (the range must then cover the whole sequence).
// KP: phase A reads a wave's K rows in KP passes (fewer passes = more loads in
// flight per wave, more registers); VU: V rows in flight per wave in phase C.
// HD: head dim, 128 or 64 (64: half the K fragments per row and half the lanes per V
// row).  DT f32: the products and sums of phase A are f32 MFMAs.
// AG, AD: the LDS arena's size (see dec::lds_arena); the exact size by default.
template <int DT, int G, int KP = 4, int VU = 8, int HD = 128, int AG = G, int AD = HD>
__device__ __forceinline__ void decode_tile(const elem_t<DT>* __restrict__ Q,
                                            const elem_t<DT>* __restrict__ K,
                                            const elem_t<DT>* __restrict__ V,
                                            elem_t<DT>* __restrict__ O, float* __restrict__ ws,
                                            uint32_t seq_len, uint32_t max_seq, uint32_t nh,
                                            uint32_t nkv, uint32_t n_split, float scale_log2,
                                            uint32_t bk, uint32_t split, uint32_t c_begin,
                                            uint32_t c_end) {
  using dec::CHUNK;
  using dec::NT;
  static_assert(HD == 128 || HD == 64, "decode head dim");
  constexpr int D = HD;
  using T = elem_t<DT>;
  constexpr int E = Vec16<DT>::kElems; // values per 16-byte load
  constexpr int NS4 = HD / (4 * E);    // 16-byte K fragments per lane and row (phase A)
  constexpr int LPR = HD / E;          // lanes per V row, E values each (phase C)
  constexpr int RG = 64 / LPR;         // V rows per wave and step
  // scores, then probabilities; rows padded by 16 floats so that phase A's 16-byte
  // writes (lane (q, g4) at row q, column 4 g4) fall in distinct banks for G <= 4
  static_assert(G <= AG && HD <= AD, "decode LDS arena");
  float* const arena = dec::lds_arena<AG, AD>();
  auto& sc = *reinterpret_cast<float(*)[G][CHUNK + 16]>(arena);
  auto& red = *reinterpret_cast<float(*)[4][G][D]>(arena + G * (CHUNK + 16));  // per-wave O
  float* const stat_m = arena + G * (CHUNK + 16) + 4 * G * D;
  float* const stat_l = stat_m + G;
  float* const stat_a = stat_l + G;

  const uint32_t b = bk / nkv, kvh = bk % nkv;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int l16 = lane & 15, g4 = lane >> 4;

  u32x4 qf[NS4];
  {
    const uint32_t hq = kvh * G + l16;
    const T* qp = Q + (static_cast<size_t>(b) * nh + hq) * D;
#pragma unroll
    for (int s = 0; s < NS4; ++s) qf[s] = (l16 < G) ? ldg128(qp + E * (4 * s + g4)) : u32x4{0, 0, 0, 0};
  }
  if (t < G) {
    stat_m[t] = -INFINITY;
    stat_l[t] = 0.0f;
  }

  float acc[G][E];
#pragma unroll
  for (int q = 0; q < G; ++q)
#pragma unroll
    for (int e = 0; e < E; ++e) acc[q][e] = 0.0f;
  const int dc = lane % LPR, rg = lane / LPR;  // phase C: d E*dc .. E*dc+E-1 of row group rg

  for (uint32_t ch = c_begin; ch < c_end; ++ch) {
    const uint32_t c0 = ch * CHUNK;
    const uint32_t n_here = (c0 < seq_len) ? min(static_cast<uint32_t>(CHUNK), seq_len - c0) : 0u;
    const T* kb = K + (static_cast<size_t>(bk) * max_seq + c0) * D;
    const T* vb = V + (static_cast<size_t>(bk) * max_seq + c0) * D;

    // ---- phase A: scores S^T = K . Q^T, 16 rows per MFMA tile ----
    {
      constexpr int TILES = CHUNK / 4 / 16;  // per wave
      constexpr int TP = TILES / KP;          // tiles whose K rows are in flight together
      static_assert(TILES % KP == 0, "K passes");
#pragma unroll
      for (int half = 0; half < KP; ++half) {
        u32x4 kf[TP][NS4];
#pragma unroll
        for (int tt = 0; tt < TP; ++tt) {
          const uint32_t row = wave * (CHUNK / 4) + (half * TP + tt) * 16 + l16;
#pragma unroll
          for (int s = 0; s < NS4; ++s) {
            const T* kp = kb + static_cast<size_t>(row) * D + E * (4 * s + g4);
            kf[tt][s] = (row < n_here) ? ldg128_nt(kp) : u32x4{0, 0, 0, 0};
          }
        }
#pragma unroll
        for (int tt = 0; tt < TP; ++tt) {
          f32x4 a4 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int s = 0; s < NS4; ++s) a4 = mfma16x16<DT>(kf[tt][s], qf[s], a4);
          const uint32_t row0 = wave * (CHUNK / 4) + (half * TP + tt) * 16 + 4 * g4;
          if (l16 < G) {
            f32x4 w;
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = (row0 + i < n_here) ? a4[i] * scale_log2 : -INFINITY;
            *reinterpret_cast<f32x4*>(&sc[l16][row0]) = w;
          }
        }
      }
    }
    __syncthreads();

    // ---- phase B: per-query max, exp, sum; merge with the running (m, l) ----
    for (int q = wave; q < G; q += 4) {
      float mx = -INFINITY;
      for (int i = lane; i < CHUNK; i += 64) mx = fmaxf(mx, sc[q][i]);
      mx = wave_max(mx);
      const float m_old = stat_m[q];
      const float m_new = fmaxf(m_old, mx);
      float sum = 0.0f;
      for (int i = lane; i < CHUNK; i += 64) {
        const float p = (m_new == -INFINITY) ? 0.0f : exp2_fast(sc[q][i] - m_new);
        sc[q][i] = p;
        sum += p;
      }
      sum = wave_sum(sum);
      if (lane == 0) {
        const float alpha = (m_old == -INFINITY) ? 0.0f : exp2_fast(m_old - m_new);
        stat_a[q] = alpha;
        stat_l[q] = stat_l[q] * alpha + sum;
        stat_m[q] = m_new;
      }
    }
    __syncthreads();

    // ---- phase C: acc = acc * alpha + sum_pos p[q][pos] * V[pos][d] ----
    {
#pragma unroll
      for (int q = 0; q < G; ++q) {
        const float a = stat_a[q];
#pragma unroll
        for (int e = 0; e < E; ++e) acc[q][e] *= a;
      }
      constexpr int ROWS_PER_WAVE = CHUNK / 4;
      constexpr int UNROLL = VU;
      static_assert((ROWS_PER_WAVE / RG) % UNROLL == 0, "V rows per pass");
#pragma unroll 1
      for (int it = 0; it < ROWS_PER_WAVE / RG; it += UNROLL) {
        u32x4 vv[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
          const uint32_t row = wave * ROWS_PER_WAVE + RG * (it + u) + rg;
          const T* vp = vb + static_cast<size_t>(row) * D + E * dc;
          vv[u] = (row < n_here) ? ldg128_nt(vp) : u32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
          const int row = wave * ROWS_PER_WAVE + RG * (it + u) + rg;
          float vf[E];
          unpack16<DT>(vv[u], vf);
#pragma unroll
          for (int q = 0; q < G; ++q) {
            const float p = sc[q][row];
#pragma unroll
            for (int e = 0; e < E; ++e) acc[q][e] = __builtin_fmaf(p, vf[e], acc[q][e]);
          }
        }
      }
    }
    __syncthreads();  // sc and stat_a are rewritten by the next chunk
  }

  // reduce the RG row groups of each wave (lanes l ^ k LPR), then the waves
#pragma unroll
  for (int q = 0; q < G; ++q)
#pragma unroll
    for (int e = 0; e < E; ++e) {
      float v = acc[q][e];
#pragma unroll
      for (int off = LPR; off < 64; off <<= 1) v += __shfl_xor(v, off);
      acc[q][e] = v;
    }
  if (rg == 0) {
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
      for (int e = 0; e < E; ++e) red[wave][q][E * dc + e] = acc[q][e];
  }
  __syncthreads();

  for (int i = t; i < G * D; i += NT) {
    const int q = i / D, d = i % D;
    const float o = red[0][q][d] + red[1][q][d] + red[2][q][d] + red[3][q][d];
    if (ws) {
      float* rec = ws + ((static_cast<size_t>(bk) * G + q) * n_split + split) * (D + 2);
      rec[2 + d] = o;
      if (d == 0) {
        rec[0] = stat_m[q];
        rec[1] = stat_l[q];
      }
    } else {
      const float l = stat_l[q];
      const float v = (l > 0.0f) ? o / l : 0.0f;
      store_elem<DT>(O + (static_cast<size_t>(b) * nh + kvh * G + q) * D + d, v);
    }
  }
  __syncthreads();  // red and stat_* are reused by the next work item
}

// Library path: n_split workgroups per (batch, kv_head), each walking `cps`
// consecutive chunks (the host picks both so that every split has at least one
// chunk).  With n_split == 1 a workgroup covers the whole sequence and writes O;
// otherwise its partial goes to the workspace for attn_decode_combine.
template <int DT, int G, int HD = 128>
__global__ void __launch_bounds__(dec::NT)
attn_decode_split(const elem_t<DT>* __restrict__ Q, const elem_t<DT>* __restrict__ K,
                  const elem_t<DT>* __restrict__ V, elem_t<DT>* __restrict__ O,
                  float* __restrict__ ws, uint32_t seq_len, uint32_t max_seq, uint32_t nh, uint32_t nkv, uint32_t n_split,
                  uint32_t cps, float scale_log2) {
  const uint32_t nchunks = (seq_len + dec::CHUNK - 1) / dec::CHUNK;
  const uint32_t split = blockIdx.x % n_split;
  const uint32_t bk = blockIdx.x / n_split;
  const uint32_t c0 = split * cps, c1 = min(nchunks, c0 + cps);
  decode_tile<DT, G, 4, 8, HD>(Q, K, V, O, n_split > 1 ? ws : nullptr, seq_len, max_seq, nh, nkv,
                               n_split, scale_log2, bk, split, c0, c1);
}

// Merge the per-chunk partials: O = sum_s 2^(m_s - M) O_s / sum_s 2^(m_s - M) l_s.
// One 512-thread block per (batch, head).  The chunk statistics (m_s, l_s) come
// in with one load per thread per 512 chunks and M is reduced over the block.
// Then four groups of 128 threads (thread d of a group owns output d) each merge
// a contiguous quarter of the chunks with sixteen O loads in flight, and the
// four partial sums are added in group order.  The merge is latency-bound (a
// few KB per head), so it is built to need few memory round trips: statistics,
// then ceil(n_split / 64) rounds of O loads.
template <int DT, int HD = 128>
__global__ void __launch_bounds__(dec::CT)
attn_decode_combine(const float* __restrict__ ws, elem_t<DT>* __restrict__ O, uint32_t nh,
                    uint32_t nkv, uint32_t n_split) {
  constexpr int D = HD, CT = dec::CT, NG = CT / D, UNR = 16;
  __shared__ float s_w[CT], s_l[CT];
  __shared__ float s_max[CT / 64];
  __shared__ float s_num[NG][D], s_den[NG][D];
  const uint32_t bhq = blockIdx.x;  // b * nh + h
  const uint32_t b = bhq / nh, h = bhq % nh;
  const uint32_t G = nh / nkv;
  const uint32_t kvh = h / G, q = h % G;
  const float* rec0 = ws + ((static_cast<size_t>(b) * nkv + kvh) * G + q) * n_split * (D + 2);
  const int t = threadIdx.x, d = t % D, grp = t / D;

  // M = max_s m_s; the first pass's (m, l) stay in registers.
  float m_own = -INFINITY, l_own = 0.0f, mx = -INFINITY;
  for (uint32_t s0 = 0; s0 < n_split; s0 += CT) {
    if (s0 + t < n_split) {
      const float m = rec0[(s0 + t) * (D + 2)];
      if (s0 == 0) {
        m_own = m;
        l_own = rec0[t * (D + 2) + 1];
      }
      mx = fmaxf(mx, m);
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
  if ((t & 63) == 0) s_max[t >> 6] = mx;
  __syncthreads();
  float M = s_max[0];
#pragma unroll
  for (int w = 1; w < CT / 64; ++w) M = fmaxf(M, s_max[w]);

  float num = 0.0f, den = 0.0f;
  for (uint32_t s0 = 0; s0 < n_split; s0 += CT) {
    const uint32_t cnt = min(static_cast<uint32_t>(CT), n_split - s0);
    if (s0 > 0) __syncthreads();  // the previous pass is done with s_w / s_l
    if (static_cast<uint32_t>(t) < cnt) {
      float m = m_own, l = l_own;
      if (s0 > 0) {
        const float* rec = rec0 + (s0 + t) * (D + 2);
        m = rec[0];
        l = rec[1];
      }
      s_w[t] = (m == -INFINITY) ? 0.0f : exp2_fast(m - M);
      s_l[t] = l;
    }
    __syncthreads();
    const uint32_t per = (cnt + NG - 1) / NG;
    const uint32_t lo = min(cnt, grp * per), hi = min(cnt, lo + per);
    const float* od = rec0 + static_cast<size_t>(s0) * (D + 2) + 2 + d;
    uint32_t i = lo;
    for (; i + UNR <= hi; i += UNR) {
      float o[UNR];
#pragma unroll
      for (int u = 0; u < UNR; ++u) o[u] = od[(i + u) * (D + 2)];
#pragma unroll
      for (int u = 0; u < UNR; ++u) {
        num = __builtin_fmaf(s_w[i + u], o[u], num);
        den = __builtin_fmaf(s_w[i + u], s_l[i + u], den);
      }
    }
    for (; i < hi; ++i) {
      num = __builtin_fmaf(s_w[i], od[i * (D + 2)], num);
      den = __builtin_fmaf(s_w[i], s_l[i], den);
    }
  }
  s_num[grp][d] = num;
  s_den[grp][d] = den;
  __syncthreads();
  if (grp == 0) {
    float n = s_num[0][d], dd = s_den[0][d];
#pragma unroll
    for (int g = 1; g < NG; ++g) {
      n += s_num[g][d];
      dd += s_den[g][d];
    }
    const float o = (dd > 0.0f) ? n / dd : 0.0f;
    store_elem<DT>(O + static_cast<size_t>(bhq) * D + d, o);
  }
}

// ============================================================================
// General attention: any head_dim <= 256, any dtype (f32 / f16 / bf16), causal
// or not.  One 256-thread workgroup per (batch, query, head); KV streamed in
// chunks of 1024 scores kept in LDS, online softmax across chunks.  Used for
// shapes outside the fast kernels.
//   kv_visible(q) = causal ? min(start_pos + q + 1, kv_len) : kv_len
// Q and O are [B][S][NH][D] (token-major) or, with head_major, [B][NH][S][D];
// kv tensors are [B][NKV][max_seq][D].
// ============================================================================
namespace gen_attn {
constexpr int CH = 1024;   // scores per pass
template <int NT>
constexpr int smem_floats() { return 256 + CH + NT / 64; }
}  // namespace gen_attn

// `smem` (LDS, gen_attn::smem_floats<NT>() floats) holds the query row, one pass of
// scores and the cross-wave reduction slots; a kernel that also runs an
// LDS-filling path passes part of that path's arena.
template <int DT, int NT = 256>
__device__ __forceinline__ void attn_general_item_smem(
    const void* __restrict__ Q, const void* __restrict__ K, const void* __restrict__ V,
    void* __restrict__ O, uint32_t seq_len, uint32_t start_pos, uint32_t max_seq,
    uint32_t kv_len, uint32_t head_dim, uint32_t nh, uint32_t nkv, int causal, float scale,
    uint32_t item, float* smem, bool head_major = false) {
  constexpr int CH = gen_attn::CH;
  constexpr int NW = NT / 64;
  static_assert(NT >= 256 && NT % 64 == 0, "head_dim up to 256 needs >= 256 threads");
  float* qs = smem;
  float* sc = smem + 256;
  float* red = smem + 256 + CH;
  const uint32_t h = item % nh;
  const uint32_t qi = (item / nh) % seq_len;
  const uint32_t b = item / (nh * seq_len);
  const uint32_t kvh = h / (nh / nkv);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  auto ld = [&](const void* p, size_t i) -> float {
    if constexpr (DT == kF32) return static_cast<const float*>(p)[i];
    else return u16_to_f32<DT>(static_cast<const uint16_t*>(p)[i]);
  };
  const size_t q_off = head_major ? ((static_cast<size_t>(b) * nh + h) * seq_len + qi) * head_dim
                                  : ((static_cast<size_t>(b) * seq_len + qi) * nh + h) * head_dim;
  const size_t kv_off = (static_cast<size_t>(b) * nkv + kvh) * max_seq * head_dim;
  for (uint32_t d = t; d < head_dim; d += NT) qs[d] = ld(Q, q_off + d);
  __syncthreads();
  const uint32_t visible = causal ? min(start_pos + qi + 1, kv_len) : kv_len;
  float m_run = -INFINITY, l_run = 0.0f, acc = 0.0f;  // acc: d = t
  for (uint32_t c0 = 0; c0 < visible; c0 += CH) {
    const uint32_t n = min(static_cast<uint32_t>(CH), visible - c0);
    for (uint32_t p = t; p < n; p += NT) {
      const size_t kr = kv_off + static_cast<size_t>(c0 + p) * head_dim;
      float dot = 0.0f;
      for (uint32_t d = 0; d < head_dim; ++d) dot = __builtin_fmaf(qs[d], ld(K, kr + d), dot);
      sc[p] = dot * scale;
    }
    __syncthreads();
    float mx = -INFINITY;
    for (uint32_t p = t; p < n; p += NT) mx = fmaxf(mx, sc[p]);
    mx = wave_max(mx);
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    mx = red[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) mx = fmaxf(mx, red[w]);
    __syncthreads();
    const float m_new = fmaxf(m_run, mx);
    const float alpha = expf(m_run - m_new);
    float sum = 0.0f;
    for (uint32_t p = t; p < n; p += NT) {
      const float e = expf(sc[p] - m_new);
      sc[p] = e;
      sum += e;
    }
    sum = wave_sum(sum);
    if (lane == 0) red[wave] = sum;
    __syncthreads();
    sum = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) sum += red[w];
    l_run = l_run * alpha + sum;
    if (static_cast<uint32_t>(t) < head_dim) {
      float a = acc * alpha;
      for (uint32_t p = 0; p < n; ++p)
        a = __builtin_fmaf(sc[p], ld(V, kv_off + static_cast<size_t>(c0 + p) * head_dim + t), a);
      acc = a;
    }
    m_run = m_new;
    __syncthreads();
  }
  if (static_cast<uint32_t>(t) < head_dim) {
    const float o = (l_run > 0.0f) ? acc / l_run : 0.0f;
    if constexpr (DT == kF32) static_cast<float*>(O)[q_off + t] = o;
    else static_cast<uint16_t*>(O)[q_off + t] = f32_to_u16<DT>(o);
  }
  __syncthreads();  // smem is reused by the next item
}

template <int DT, int NT = 256>
__device__ __forceinline__ void attn_general_item(
    const void* __restrict__ Q, const void* __restrict__ K, const void* __restrict__ V,
    void* __restrict__ O, uint32_t seq_len, uint32_t start_pos, uint32_t max_seq,
    uint32_t kv_len, uint32_t head_dim, uint32_t nh, uint32_t nkv, int causal, float scale,
    uint32_t item) {
  __shared__ float smem[gen_attn::smem_floats<NT>()];
  attn_general_item_smem<DT, NT>(Q, K, V, O, seq_len, start_pos, max_seq, kv_len, head_dim, nh,
                                 nkv, causal, scale, item, smem);
}

template <int DT>
__global__ void __launch_bounds__(256)
attn_general(const void* __restrict__ Q, const void* __restrict__ K, const void* __restrict__ V,
             void* __restrict__ O, uint32_t batch, uint32_t seq_len, uint32_t start_pos,
             uint32_t max_seq, uint32_t kv_len, uint32_t head_dim, uint32_t nh, uint32_t nkv,
             int causal, float scale) {
  (void)batch;
  attn_general_item<DT>(Q, K, V, O, seq_len, start_pos, max_seq, kv_len, head_dim, nh, nkv,
                        causal, scale, blockIdx.x);
}

// Causal mask on an f32 tile (mlir_to_linalg.rs:1191-1247): y = x where col <= row,
// else -inf.  Bit-exact.  Rows are `rows` long tiles stacked `tiles` deep.
__global__ void __launch_bounds__(256)
causal_mask_f32(const float* __restrict__ x, float* __restrict__ y, uint32_t rows, uint32_t cols,
                uint64_t total) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= total) return;
  const uint32_t c = static_cast<uint32_t>(i % cols);
  const uint32_t r = static_cast<uint32_t>((i / cols) % rows);
  y[i] = (c <= r) ? x[i] : __uint_as_float(0xff800000u);
}

}  // namespace th
