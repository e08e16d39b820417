// f32 attention on the fp32 matrix cores (v_mfma_f32_32x32x2_f32): single-head below,
// causal GQA prefill further down.
//
// Single-head, non-causal attention on S x D tiles: the __tile_attention_f32 op (crates/tile_std/src/
// tile.rs:221, :2401; linalg semantics crates/rustc_codegen_tile/src/
// mlir_to_linalg.rs:1781-1902: O = softmax(Q K^T * scale) V, scale = 1/sqrt(D)
// rounded from f64 to f32).
//
// Flash form: one 256-thread workgroup per (tile, 128-query block), 32 queries
// per wave; K and V stream through LDS in blocks of 32 positions (two buffers,
// the next block prefetched into registers while the current one computes), and
// the softmax runs online with f32 row max and sum.
//
// Per 32-position block a wave computes S^T = K . Q^T as one 32 x 32 MFMA block:
// the A operand is K (lane l: position l % 32), the B operand Q^T lives in
// registers for the whole pass (lane l: query l % 32), so accumulator r of lane l
// is the score of query l % 32 at position f(r, h) = 8 (r / 4) + 4 h + r % 4,
// h = l / 32.  The row max needs one exchange between the lane halves.  The
// probabilities then feed O += P . V without moving: step r of the 16 MFMA steps
// takes position f(r, h) from lane half h, for P (A operand, registers) and V
// (B operand, LDS row f(r, h)) alike.  O's accumulator rows are queries, so the
// per-query rescale factors and final sums go through a 32-float LDS slot per
// wave.  The head dimension is split between lane halves in the S^T product as
// d = 4 (ks / 2) + 2 h + ks % 2, so a lane's K values for steps 2m and 2m+1 are
// adjacent (one 8-byte LDS read) and its Q^T registers fill from 16-byte loads of
// its query row.  In O += P . V, 32-column block c of O holds head dims
// d = ND n + c (n = l32, ND = D / 32 blocks), so a lane reads its V values for all
// blocks as ND adjacent floats (one 16-byte read at D 128) and writes its O row
// piece as one 16-byte store.
//
// LDS rows: K [32][D + 2] (an 8-byte read of positions 0..31 covers the 64 banks
// once per lane half), V [32][D] (each 16-byte read takes 128 contiguous bytes per
// eight lanes).  Reading K and V one float per lane, paired by the compiler into
// two-address reads, cost one bank-conflict cycle per MFMA (27% of LDS-active
// cycles).
//
// Work order: the 128-query blocks of one problem run on one XCD, so its K and V
// are read from HBM about once and then served by that XCD's L2.
#pragma once

#include "attention.hpp"
#include "common.hpp"

namespace th {
namespace af32 {
constexpr int BQ = 128;   // queries per workgroup
constexpr int BKV = 32;   // positions per K/V block
constexpr int NT = 256;

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// 16-byte aligned: V tiles go in, and the per-wave factors come out, as 16-byte LDS
// accesses
template <int D>
struct alignas(16) Lds {
  float k[2][BKV * (D + 2)];
  float v[2][BKV * D];
  float stat[NT / 64][32];   // per-wave query factors (rescale, then 1 / sum)
};
template <int D>
__device__ __forceinline__ Lds<D>& smem() {
  __shared__ Lds<D> s;
  return s;
}
}  // namespace af32

// Queries qb*128 .. +127 of problem `tile` (Q, K, V, O: [tiles][S][D] f32).
template <int D>
__device__ __forceinline__ void attn_f32_tile(const float* __restrict__ Q,
                                              const float* __restrict__ K,
                                              const float* __restrict__ V, float* __restrict__ O,
                                              uint32_t S, float scale_log2, uint32_t tile,
                                              uint32_t qb) {
  using namespace af32;
  static_assert(D == 64 || D == 128, "head_dim 64 or 128");
  constexpr int LK = D + 2, LV = D;
  constexpr int KP = BKV * D / 2 / NT;   // float2 pieces of K per thread
  constexpr int VP = BKV * D / 4 / NT;   // float4 pieces of V per thread
  constexpr int ND = D / 32;             // 32-wide column blocks of O
  Lds<D>& s = smem<D>();
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int h = lane >> 5, l32 = lane & 31;
  const size_t base = static_cast<size_t>(tile) * S * D;
  const float* Kt = K + base;
  const float* Vt = V + base;

  // Q^T operand: q = q0 + 32 wave + l32 (rows past S read row S-1, not stored)
  const uint32_t q = qb * BQ + 32 * wave + l32;
  const uint32_t qc = min(q, S - 1);
  float qf[D / 2];
  {
    const float* qr = Q + base + static_cast<size_t>(qc) * D;
#pragma unroll
    for (int j = 0; j < D / 4; ++j) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(qr + 4 * j);
      qf[2 * j] = x[2 * h];
      qf[2 * j + 1] = x[2 * h + 1];
    }
  }

  f32x2 rk[KP];
  f32x4 rv[VP];
  auto load = [&](uint32_t kv0) {
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const int e = t + NT * i;               // piece e: row e / (D/2), cols 2 (e % (D/2))
      const uint32_t row = kv0 + e / (D / 2);
      rk[i] = row < S ? *reinterpret_cast<const f32x2*>(Kt + static_cast<size_t>(row) * D + 2 * (e % (D / 2)))
                      : f32x2{0.0f, 0.0f};
    }
#pragma unroll
    for (int i = 0; i < VP; ++i) {
      const int e = t + NT * i;
      const uint32_t row = kv0 + e / (D / 4);
      rv[i] = row < S ? *reinterpret_cast<const f32x4*>(Vt + static_cast<size_t>(row) * D + 4 * (e % (D / 4)))
                      : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const int e = t + NT * i;
      *reinterpret_cast<f32x2*>(&s.k[buf][(e / (D / 2)) * LK + 2 * (e % (D / 2))]) = rk[i];
    }
#pragma unroll
    for (int i = 0; i < VP; ++i) {
      const int e = t + NT * i;
      *reinterpret_cast<f32x4*>(&s.v[buf][(e / (D / 4)) * LV + 4 * (e % (D / 4))]) = rv[i];
    }
  };

  f32x16 acc[ND];
#pragma unroll
  for (int c = 0; c < ND; ++c)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[c][r] = 0.0f;
  float m_run = -INFINITY, l_run = 0.0f;   // of query l32 (l_run: this half's share)

  const uint32_t nb = (S + BKV - 1) / BKV;
  load(0);
  store(0);
  __syncthreads();
  for (uint32_t jb = 0; jb < nb; ++jb) {
    const int cur = jb & 1;
    if (jb + 1 < nb) load((jb + 1) * BKV);
    // ---- S^T = K . Q^T ----
    f32x16 st;
#pragma unroll
    for (int r = 0; r < 16; ++r) st[r] = 0.0f;
    const float* kr = s.k[cur] + l32 * LK + 2 * h;
#pragma unroll
    for (int m = 0; m < D / 4; ++m) {
      const f32x2 k2 = *reinterpret_cast<const f32x2*>(kr + 4 * m);
      st = __builtin_amdgcn_mfma_f32_32x32x2f32(k2[0], qf[2 * m], st, 0, 0, 0);
      st = __builtin_amdgcn_mfma_f32_32x32x2f32(k2[1], qf[2 * m + 1], st, 0, 0, 0);
    }
    // ---- online softmax of query l32 over positions f(r, h) ----
    const uint32_t kv0 = jb * BKV;
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const uint32_t pos = kv0 + 8 * (r >> 2) + 4 * h + (r & 3);
      st[r] = pos < S ? st[r] * scale_log2 : -INFINITY;
      mx = fmaxf(mx, st[r]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m_run, mx);    // finite: every block has a position < S
    const float alpha = exp2_fast(m_run - m_new);
    float sum = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      st[r] = exp2_fast(st[r] - m_new);
      sum += st[r];
    }
    l_run = l_run * alpha + sum;
    m_run = m_new;
    // ---- O = O * alpha + P . V (O rows are queries: alpha through LDS) ----
    if (h == 0) s.stat[wave][l32] = alpha;
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): the wave's own LDS write
    __builtin_amdgcn_wave_barrier();
    {
      const f32x4* sa = reinterpret_cast<const f32x4*>(&s.stat[wave][4 * h]);
      f32x4 a4[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) a4[g] = sa[2 * g];   // queries 8 g + 4 h .. +3
#pragma unroll
      for (int c = 0; c < ND; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[c][r] *= a4[r >> 2][r & 3];
    }
    const float* vr = s.v[cur] + (4 * h) * LV + ND * l32;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float* vrow = vr + (8 * (r >> 2) + (r & 3)) * LV;
      float vv[ND];
      if constexpr (ND == 4) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(vrow);
#pragma unroll
        for (int c = 0; c < 4; ++c) vv[c] = x[c];
      } else {
        const f32x2 x = *reinterpret_cast<const f32x2*>(vrow);
        vv[0] = x[0];
        vv[1] = x[1];
      }
#pragma unroll
      for (int c = 0; c < ND; ++c)
        acc[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(st[r], vv[c], acc[c], 0, 0, 0);
    }
    if (jb + 1 < nb) store(cur ^ 1);
    __syncthreads();   // also orders this block's stat reads before the next writes
  }

  // ---- O / l, rows of the accumulator are queries 8 (r / 4) + 4 h + r % 4 ----
  const float l_tot = l_run + __shfl_xor(l_run, 32);
  if (h == 0) s.stat[wave][l32] = 1.0f / l_tot;
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_wave_barrier();
  const uint32_t qw = qb * BQ + 32 * wave;
  const bool o16 = (reinterpret_cast<uintptr_t>(O) & 15) == 0;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int qi = 8 * (r >> 2) + 4 * h + (r & 3);
    const float inv = s.stat[wave][qi];
    if (qw + qi < S) {
      // columns ND l32 .. ND l32 + ND - 1 of the row
      float* orow = O + base + static_cast<size_t>(qw + qi) * D + ND * l32;
      f32x4 ov;
#pragma unroll
      for (int c = 0; c < 4; ++c) ov[c] = c < ND ? acc[c < ND ? c : 0][r] * inv : 0.0f;
      if (ND == 4 && o16) {
        *reinterpret_cast<f32x4*>(orow) = ov;
      } else {
#pragma unroll
        for (int c = 0; c < ND; ++c) orow[c] = ov[c];
      }
    }
  }
  __syncthreads();   // LDS is reused by the next work item
}

namespace af32 {
// Work item of hardware block `bid` out of `total`: the hardware deals workgroups
// to the 8 XCDs round-robin, so item ids are renumbered to give each XCD a
// contiguous run (consecutive query blocks of one problem share its L2).
__device__ __forceinline__ uint32_t xcd_item(uint32_t bid, uint32_t total) {
  return total % 8 == 0 ? (bid % 8) * (total / 8) + bid / 8 : bid;
}
}  // namespace af32

// Library kernel: grid = tiles * ceil(S / 128), S >= 1.
template <int D>
__global__ void __launch_bounds__(af32::NT)
attn_f32_mfma(const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
              float* __restrict__ O, uint32_t S, float scale_log2) {
  const uint32_t nqb = (S + af32::BQ - 1) / af32::BQ;
  const uint32_t w = af32::xcd_item(blockIdx.x, gridDim.x);
  attn_f32_tile<D>(Q, K, V, O, S, scale_log2, w / nqb, w % nqb);
}

// ============================================================================
// Causal GQA prefill on f32 (__tile_attention_prefill_f32: crates/tile_std/src/
// tile.rs:2136, :3064; Metal template mlir_to_msl.rs:10928-11009), head_dim 64/128.
//
// Bound: the fp32 matrix cores (4 D FLOP per query and visible position).  One
// 256-thread workgroup per (batch, head, 64 queries): wave (g, kh) = (w / 2, w % 2)
// takes queries 32 g .. +31 against the 32-position half kh of every 64-position
// stage, and the two halves' (m, l, O) merge through LDS at the end.  64 queries
// rather than attn_f32_tile's 128 double the work items, so a prompt of 1000 tokens
// fills the chip (512 items for 32 heads, two per CU), and the causal triangle wastes
// at most half as many masked scores.
//
// K and V each have one stage buffer (32 KB at D 128, so two workgroups share a CU),
// filled by LDS DMA: K(j+1) is issued when every wave has read K(j) and lands under
// the softmax and P.V of stage j; V(j+1) is issued when every wave has read V(j) and
// lands under the scores of stage j+1.  Operand layouts are attn_f32_tile's, except
// that the head dimension is split d = 8 m + 4 h + j, so K comes in with 16-byte
// reads; chunk c of K row r sits at c ^ (r % chunks per row) (conflict-free).
//
// A position above a query's diagonal contributes nothing, also when its V row holds
// infinities or NaN: in the one stage half that crosses the diagonal V enters the
// MFMA with those values zeroed, and they are added for the queries that see them.
//
// Measured on MI355X, 1001 queries of 32 heads over 8 kv heads, D 128: 92.9 us (88 TFLOP/s
// of the fp32 matrix cores' 157) against 7376 us on the general kernel, a workgroup per query
// with scalar loads.
// ============================================================================
namespace pf32 {
constexpr int BQ = 64;    // queries per workgroup
constexpr int BKV = 64;   // positions per stage (two wave halves of 32)
constexpr int NT = 256;
using af32::f32x2;

template <int D>
struct alignas(16) Lds {
  float k[BKV * D];
  float v[BKV * D];
  float stat[4][2][32];   // per wave: query factors, then (m, l)
};
}  // namespace pf32

// Queries qb*64 .. +63 of head h, batch b.  Q, O: [B][S][nh][D]; K, V: [B][nkv][max_seq][D].
template <int D>
__device__ __forceinline__ void prefill_f32_tile(const float* __restrict__ Q,
                                                 const float* __restrict__ K,
                                                 const float* __restrict__ V,
                                                 float* __restrict__ O, uint32_t S,
                                                 uint32_t start_pos, uint32_t max_seq, uint32_t nh,
                                                 uint32_t nkv, float scale_log2, uint32_t b,
                                                 uint32_t head, uint32_t qb) {
  using namespace pf32;
  static_assert(D == 64 || D == 128, "head_dim 64 or 128");
  constexpr int ND = D / 32;        // 32-wide column blocks of O
  constexpr int CPR = D / 4;        // 16-byte chunks per row
  constexpr int RPU = 64 / CPR;     // rows per 1 KB DMA unit
  constexpr int UPW = BKV / RPU / 4;   // DMA units per wave and operand
  __shared__ Lds<D> s;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int h = lane >> 5, l32 = lane & 31;
  const int g = wave >> 1, kh = wave & 1;
  const uint32_t kv_len = start_pos + S;
  const size_t kvo = (static_cast<size_t>(b) * nkv + head / (nh / nkv)) * max_seq * D;
  const uint32_t q0 = qb * BQ;
  const uint32_t nst = (start_pos + min(q0 + BQ, S) + BKV - 1) / BKV;

  // DMA of a stage: lane i of unit u fills slot i % CPR of row RPU u + i / CPR; rows past
  // the last position read that position's row (masked for every query)
  auto issue = [&](const float* src, float* dst, uint32_t j, bool swz) {
    const float* base = src + kvo + static_cast<size_t>(j) * BKV * D;
    const int last = static_cast<int>(kv_len - 1 - j * BKV);
    int drow = wave * UPW * RPU + lane / CPR, dslot = lane % CPR;
    asm volatile("" : "+v"(drow), "+v"(dslot));   // recomputed per stage: registers are short
#pragma unroll
    for (int i = 0; i < UPW; ++i) {
      const int row = drow + i * RPU;
      const int c = swz ? dslot ^ (row & (CPR - 1)) : dslot;
      lds::dma16(base + static_cast<uint32_t>(min(row, last) * D + 4 * c),
                 dst + (wave * UPW + i) * 256);
    }
  };
  issue(K, s.k, 0, true);
  issue(V, s.v, 0, false);

  // Q^T operand: query qw + l32 (rows past S read row S - 1, not stored)
  const uint32_t qw = q0 + 32 * g;
  const uint32_t qc = min(qw + l32, S - 1);
  float qf[D / 2];
  {
    const float* qr = Q + ((static_cast<size_t>(b) * S + qc) * nh + head) * D + 4 * h;
#pragma unroll
    for (int m = 0; m < D / 8; ++m) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(qr + 8 * m);
#pragma unroll
      for (int j = 0; j < 4; ++j) qf[4 * m + j] = x[j];
    }
  }
  const uint32_t vis = start_pos + qc + 1;   // positions [0, vis) are visible

  f32x16 acc[ND];
#pragma unroll
  for (int c = 0; c < ND; ++c)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[c][r] = 0.0f;
  float m_run = -INFINITY, l_run = 0.0f;   // of query l32 (l_run: this lane half's share)

  const int krow = 32 * kh + l32;
  const uint32_t kbase = krow * CPR + (h ^ (krow & (CPR - 1)));   // in 16-byte chunks
  const uint32_t vbase = (32 * kh + 4 * h) * D + ND * l32;

  for (uint32_t j = 0; j < nst; ++j) {
    const uint32_t kv0 = j * BKV + 32 * kh;
    const bool live = qw < S && kv0 < start_pos + min(qw + 32, S);   // some query sees some position
    const bool diag = kv0 + 32 > start_pos + qw + 1;                 // some query misses one
    lds::wait_vm<UPW>();   // K(j) landed; V(j) may be in flight
    lds::bar();
    f32x16 st;
#pragma unroll
    for (int r = 0; r < 16; ++r) st[r] = 0.0f;
    if (live) {
      // ---- S^T = K . Q^T: each read one group of four MFMAs ahead of its use ----
      const f32x4* k4 = reinterpret_cast<const f32x4*>(s.k);
      uint32_t kb = kbase;
      asm volatile("" : "+v"(kb));   // the D / 8 addresses are not kept across stages
      f32x4 nxt = k4[kb];
#pragma unroll
      for (int m = 0; m < D / 8; ++m) {
        const f32x4 cur = nxt;
        if (m + 1 < D / 8) nxt = k4[kb ^ (2 * m + 2)];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          st = __builtin_amdgcn_mfma_f32_32x32x2f32(cur[i], qf[4 * m + i], st, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    lds::wait_lgkm0();
    lds::bar();   // every wave has read K(j)
    if (j + 1 < nst) issue(K, s.k, j + 1, true);
    if (live) {
      // ---- online softmax of query l32 over positions kv0 + f(r, h) ----
      float mx = -INFINITY;
      if (diag) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const uint32_t pos = kv0 + 8 * (r >> 2) + 4 * h + (r & 3);
          st[r] = pos < vis ? st[r] * scale_log2 : -INFINITY;
          mx = fmaxf(mx, st[r]);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          st[r] *= scale_log2;
          mx = fmaxf(mx, st[r]);
        }
      }
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float m_new = fmaxf(m_run, mx);
      // nothing finite so far (masked, or scores of -inf): every p is 2^-inf = 0
      const float m_sub = m_new == -INFINITY ? 0.0f : m_new;
      const float alpha = exp2_fast(m_run - m_sub);
      float sum = 0.0f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        st[r] = exp2_fast(st[r] - m_sub);
        sum += st[r];
      }
      l_run = l_run * alpha + sum;
      m_run = m_new;
      // ---- O = O * alpha (O rows are queries: alpha through LDS) ----
      if (__ballot(alpha != 1.0f)) {
        if (h == 0) s.stat[wave][0][l32] = alpha;
        lds::wait_lgkm0();
        __builtin_amdgcn_wave_barrier();
        const f32x4* sa = reinterpret_cast<const f32x4*>(&s.stat[wave][0][4 * h]);
        f32x4 a4[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) a4[i] = sa[2 * i];   // queries 8 i + 4 h .. +3
#pragma unroll
        for (int c = 0; c < ND; ++c)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[c][r] *= a4[r >> 2][r & 3];
      }
    }
    if (j + 1 < nst) lds::wait_vm<UPW>();   // V(j) landed; K(j+1) may be in flight
    else lds::wait_vm<0>();
    lds::bar();
    if (live) {
      // ---- O += P . V ----
      // each read one group of ND MFMAs ahead of its use
      typedef float vecv __attribute__((ext_vector_type(ND)));
      auto load_v = [&](int r) {
        return *reinterpret_cast<const vecv*>(&s.v[vbase + (8 * (r >> 2) + (r & 3)) * D]);
      };
      bool bad = false;
      auto pv = [&](auto clean) {
        vecv nxt = load_v(0);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          vecv cur = nxt;
          if (r + 1 < 16) nxt = load_v(r + 1);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int c = 0; c < ND; ++c) {
            float x = cur[c];
            if constexpr (decltype(clean)::value) {
              const bool fin = fabsf(x) < INFINITY;
              bad |= !fin;
              x = fin ? x : 0.0f;
            }
            acc[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(st[r], x, acc[c], 0, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      if (!diag) {
        pv(std::false_type{});
      } else {
        pv(std::true_type{});
        if (__ballot(bad)) {
          // the infinities and NaN left out above, for the queries that see their position
#pragma unroll 1
          for (int p = 0; p < 32; ++p) {
            const int rp = 4 * (p >> 3) + (p & 3), hp = (p >> 2) & 1;   // p = f(rp, hp)
            float ps = st[0];
#pragma unroll
            for (int r = 1; r < 16; ++r) ps = rp == r ? st[r] : ps;
            if (h == hp) s.stat[wave][0][l32] = ps;
            lds::wait_lgkm0();
            __builtin_amdgcn_wave_barrier();
            const f32x4* sp = reinterpret_cast<const f32x4*>(&s.stat[wave][0][4 * h]);
#pragma unroll
            for (int c = 0; c < ND; ++c) {
              const float x = s.v[(32 * kh + p) * D + ND * l32 + c];
              const bool inf = !(fabsf(x) < INFINITY);
#pragma unroll
              for (int r = 0; r < 16; ++r) {
                const uint32_t qi = 8 * (r >> 2) + 4 * h + (r & 3);
                const float a = __builtin_fmaf(sp[2 * (r >> 2)][r & 3], x, acc[c][r]);
                acc[c][r] = inf && kv0 + p <= start_pos + qw + qi ? a : acc[c][r];
              }
            }
            lds::wait_lgkm0();
            __builtin_amdgcn_wave_barrier();
          }
        }
      }
    }
    lds::wait_lgkm0();
    lds::bar();   // every wave has read V(j)
    if (j + 1 < nst) issue(V, s.v, j + 1, false);
  }

  // ---- merge the two position halves (the stage buffers are idle: K(nst) was not issued) ----
  const float l_half = l_run + __shfl_xor(l_run, 32);
  if (kh == 1) {
    float* x = (g == 0) ? s.k : s.v;   // 16 KB (8 KB at D 64) each: ND * 16 rows of 64 lanes
#pragma unroll
    for (int c = 0; c < ND; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r) x[(16 * c + r) * 64 + lane] = acc[c][r];
    if (h == 0) {
      s.stat[wave][0][l32] = m_run;
      s.stat[wave][1][l32] = l_half;
    }
  }
  __syncthreads();
  if (kh == 0 && qw < S) {
    const float m1 = s.stat[wave + 1][0][l32], l1 = s.stat[wave + 1][1][l32];
    const float M = fmaxf(m_run, m1);
    const float f0 = m_run == -INFINITY ? 0.0f : exp2_fast(m_run - M);
    const float f1 = m1 == -INFINITY ? 0.0f : exp2_fast(m1 - M);
    const float l = l_half * f0 + l1 * f1;
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    __builtin_amdgcn_wave_barrier();
    if (h == 0) {
      s.stat[wave][0][l32] = f0 * inv;
      s.stat[wave][1][l32] = f1 * inv;
    }
    lds::wait_lgkm0();
    __builtin_amdgcn_wave_barrier();
    const float* x = (g == 0) ? s.k : s.v;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int qi = 8 * (r >> 2) + 4 * h + (r & 3);
      const float a0 = s.stat[wave][0][qi], a1 = s.stat[wave][1][qi];
      if (qw + qi >= S) continue;
      float ov[ND];
#pragma unroll
      for (int c = 0; c < ND; ++c) {
        // a half that saw nothing has factor 0 and O 0; a sum that is not positive gives 0
        const float o = acc[c][r] * a0 + x[(16 * c + r) * 64 + lane] * a1;
        ov[c] = a0 + a1 > 0.0f ? o : 0.0f;
      }
      // columns ND l32 .. +ND - 1 of the row
      float* orow = O + ((static_cast<size_t>(b) * S + qw + qi) * nh + head) * D + ND * l32;
      if constexpr (ND == 4) *reinterpret_cast<f32x4*>(orow) = f32x4{ov[0], ov[1], ov[2], ov[3]};
      else *reinterpret_cast<f32x2*>(orow) = f32x2{ov[0], ov[1]};
    }
  }
}

// Work index of workgroup w of `total` on a device of `cus` CUs.  The second workgroup of a CU
// runs beside the one `cus` before it: heavy first in both rounds would give one CU the
// heaviest items of each.  So the second round runs light first (its XCD order kept).
// Measured on MI355X, 32 heads over 8, us with both rounds heavy first and now: 1001 queries
// (512 items) 114.4 -> 91.7, D 64 63.4 -> 52.6; 640 (320) 64.5 -> 61.4; 1000 after 1024 250 ->
// 225; later rounds stay heavy first: 1536 (768) 188 -> 190, D 64 102 -> 104; 2048 (1024) 332
// -> 306, D 64 181 -> 167; 4096 (2048) 1164 -> 1155, D 64 630 -> 626.  Every odd round light
// first: 2048 329, 4096 1173; rounds of two per CU: 1536 213, 2048 369, 4096 1148.
__device__ __forceinline__ uint32_t prefill_f32_item(uint32_t w, uint32_t total, uint32_t cus) {
  if (w / cus != 1) return w;
  const uint32_t n = min(cus, total - cus), l = w - cus;
  const uint32_t step = total % 8 == 0 && cus % 8 == 0 ? 8 : 1;
  return cus + (n / step - 1 - l / step) * step + l % step;
}

// Library kernel: grid = batch * nh * ceil(S / 64), S >= 1; heavy query blocks first (but for
// the second round: prefill_f32_item), a kv head's query blocks on one XCD (prefill_work).
template <int D>
__global__ void __launch_bounds__(pf32::NT, 2)
attn_prefill_f32(const float* __restrict__ Q, const float* __restrict__ K,
                 const float* __restrict__ V, float* __restrict__ O, uint32_t batch, uint32_t S,
                 uint32_t start_pos, uint32_t max_seq, uint32_t nh, uint32_t nkv,
                 float scale_log2, uint32_t cus) {
  uint32_t bh, qb;
  prefill_work(prefill_f32_item(blockIdx.x, gridDim.x, cus), batch, nh, nkv,
               (S + pf32::BQ - 1) / pf32::BQ, bh, qb);
  prefill_f32_tile<D>(Q, K, V, O, S, start_pos, max_seq, nh, nkv, scale_log2, bh / nh, bh % nh,
                      qb);
}

}  // namespace th
