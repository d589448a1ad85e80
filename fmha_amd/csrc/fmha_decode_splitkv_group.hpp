// fmha_decode_splitkv_group.hpp -- the split-KV scores pass on the matrix
// cores, for query groups of 8 and more (lengths beyond 16 rows), and two
// single passes.
//
// The VALU scores pass (fmha_decode_splitkv.hpp) spends per lane about G * D
// / 8 multiply-adds per row, so its time grows with G: the host runs a group
// above 8 on it as ceil(G / 8) launch KV heads of 8 query heads
// (SplitArgs::kv_groups).  Here the products are MFMAs over 16-column tiles
// of query heads, as in fmha_decode_group.hpp, and one wave serves one KV
// head with all of its query heads: it takes HPW = 64 / (D/8) consecutive
// 16-row blocks of one (batch, KV head), one block per lane group, loads
// their K rows as the VALU pass does (LongRows, rows past the length read as
// 0) and stages them in LDS; per 16-column tile of query heads (B operand
// read straight from Q in the MFMA's layout) and block, S^T = K_blk . Q^T is
// D/32 v_mfma_f32_16x16x32_bf16.  The scaled scores and the statistics of
// the workgroup's rows go to the same workspace arrays as the VALU pass's;
// the P.V launch (fmha_decode_splitkv_pv.hpp) is shared.
//
// Packed and strided layouts read rows through LongRows' one descriptor per
// wave; on paged layouts the lane groups of a wave read rows of different
// pages, which one page's descriptor cannot cover, so PagedLaneRows gives
// every lane its own 64-bit addresses instead.  The query heads of a KV head
// may be padded (Q and O copies with a multiple of 8 heads): the kernels
// take G = num_heads_q / num_heads_kv as given.
//
// The file ends with two single passes on the same products (one launch,
// nothing through the workspace) for query groups of at most 16 with
// enough (batch, KV head) units: onepass_mfma_kernel, one workgroup per
// unit keeping the row's scores in LDS, and onepass_mfma_reg_kernel, each
// wave of the workgroup keeping its rows' scores in the registers the
// scores MFMA leaves them in.
#pragma once

#include "fmha_decode_group.hpp"
#include "fmha_decode_splitkv.hpp"

namespace fmha_decode {

// The row loader of the matrix-core split passes for a layout: per-lane
// addresses on every paged layout.
template <int D, int LAYOUT>
using GroupRows = typename std::conditional<
    is_paged_layout(LAYOUT), PagedLaneRows<D, LAYOUT == kLayoutPagedBlock || LAYOUT == kLayoutPagedBlockLanes>,
    LongRows<D, LAYOUT>>::type;

// Grid: pieces (batch_piece) of 2^sup_shift rows, HPW blocks, times Hkv
// one-wave workgroups, piece * Hkv + hk (consecutive ones: neighbouring heads
// of the same rows).
template <int D, int LAYOUT>
__global__ __launch_bounds__(kBlockThreads) void splitkv_scores_group_kernel(SplitArgs a) {
  using Sh = GroupShape<D>;
  constexpr int LPH = Sh::LPH;
  constexpr int HPW = Sh::HPW;
  constexpr int NR = kSplitBlockRows;
  __shared__ __attribute__((aligned(16))) char k_lds[NR * Sh::KS];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const uint32_t hkv = (uint32_t)a.num_heads_kv;
  const uint32_t u = blockIdx.x / hkv;
  const uint32_t hk = blockIdx.x - u * hkv;
  RowPiece rp;
  if (!batch_piece<LAYOUT>(a, u, a.sup_shift, (uint32_t)a.nsup, rp)) return;
  const uint32_t b = rp.b;
  const int S = rp.S;
  const int hq = a.num_heads_q;
  const int G = hq / (int)hkv;
  const int tiles = (G + 15) / 16;
  const int64_t row_base = split_row_base<LAYOUT>(a, b);  // ahead of clear_done's stores (splitkv_scores_kernel)
  if (rp.piece == 0) clear_done(a, b, hk, 1, tiles * a.pv.parts);
  if (S <= 0 || S > a.max_rows) return;
  const int j0 = (int)(rp.piece << a.sup_shift);  // the wave's first row
  const int s = lane / LPH;  // this lane group's block of the wave
  const int r = lane % LPH;
  const int q = lane >> 4;   // MFMA lane group
  const int n = lane & 15;   // MFMA row / column

  // K rows of the wave's blocks (lane group s: rows j0 + 16 s + j).
  GroupRows<D, LAYOUT> kv;
  kv.init(a, a.k, b, row_base, 0, S, (int)hk, true, r, s * NR);
  u32x4 kr[NR];
  kv.template load<NR>(kr, j0);
  const bool kv_bad = kv.any_bad();
  // This KV head's query rows: tile t's B operands (lane (q, n): query
  // column 16 t + n, 16-byte chunks 4 cc + q), requested one tile ahead.
  const __amdgpu_buffer_rsrc_t q_rsrc =
      make_rsrc(a.q + ((uint64_t)b * hq + (uint64_t)hk * G) * D, (uint32_t)G * D * 2u);
  auto load_q = [&](bf16x8_v (&dst)[Sh::QLD], int tile) {
    const int g = tile * 16 + n;
#pragma unroll
    for (int cc = 0; cc < Sh::QLD; ++cc)
      dst[cc] = __builtin_bit_cast(
          bf16x8_v, buffer_load16<kPolicyDefault>(q_rsrc, g < G && tile < tiles
                                                              ? (uint32_t)(g * D + (4 * cc + q) * 8) * 2u
                                                              : kLaneOutOfRange));
  };
  bf16x8_v qn[Sh::QLD];
  load_q(qn, 0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < NR; ++j) *reinterpret_cast<u32x4*>(k_lds + j * Sh::KS + s * D * 2 + r * 16) = kr[j];
  wave_lds_sync();

  // The scores of the wave's blocks.
  const int blk0 = j0 / NR;
  const int nb = a.nblk - blk0 < HPW ? a.nblk - blk0 : HPW;
  const __amdgpu_buffer_rsrc_t t_rsrc =
      make_rsrc(a.t + t_block_base(a, b, blk0), (uint32_t)nb * (uint32_t)hq * NR * 4u);
  for (int tile = 0; tile < tiles; ++tile) {
    const int g = tile * 16 + n;  // this lane's query column
    const bool gok = g < G;
    bf16x8_v qb[Sh::QLD];
#pragma unroll
    for (int cc = 0; cc < Sh::QLD; ++cc) qb[cc] = qn[cc];
    if (tile + 1 < tiles) load_q(qn, tile + 1);
    float x[HPW][4];
    float m = -__builtin_inff();  // this lane's rows of the column
#pragma unroll
    for (int p = 0; p < HPW; ++p) {
      const int jb = j0 + p * NR;  // first row of block p
      if (jb >= S) break;
      f32x4_v c4 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int cc = 0; cc < Sh::QLD; ++cc) {
        const bf16x8_v ka = *reinterpret_cast<const bf16x8_v*>(k_lds + n * Sh::KS + p * D * 2 + (4 * cc + q) * 16);
        c4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, qb[cc], c4, 0, 0, 0);
      }
      // Rows 4q..4q+3 of block p for query column g.
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[p][e] = c4[e] * a.scale;
        m = jb + 4 * q + e < S ? fmaxf(m, x[p][e]) : m;
      }
      // Scores of rows past S (their K rows read as 0) land in the block's
      // padding, which nothing reads as a weight.
      if (gok) {
        const u32x4 v4 = {__builtin_bit_cast(uint32_t, x[p][0]), __builtin_bit_cast(uint32_t, x[p][1]),
                          __builtin_bit_cast(uint32_t, x[p][2]), __builtin_bit_cast(uint32_t, x[p][3])};
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_gcc, v4), t_rsrc,
                                               (int)((((uint32_t)p * hq + hk * G + g) * NR + 4 * q) * 4u), 0,
                                               kPolicyStreamStore);
      }
    }
    // The column's max and sum of exponentials over the wave's rows (row j0
    // is valid, so the max is finite for finite scores).
    m = column_reduce<true>(m);
    float l = 0.0f;
#pragma unroll
    for (int p = 0; p < HPW; ++p) {
      const int jb = j0 + p * NR;
      if (jb >= S) break;
#pragma unroll
      for (int e = 0; e < 4; ++e) l += jb + 4 * q + e < S ? expf(x[p][e] - m) : 0.0f;
    }
    l = column_reduce<false>(l);
    // An unmapped page among the wave's rows: a NaN sum makes the batch's
    // weights, hence its outputs, NaN.
    if (q == 0 && gok)
      a.st[((uint64_t)b * hq + (uint64_t)hk * G + g) * a.nsup + rp.piece] =
          f32x2_v{m, kv_bad ? __builtin_nanf("") : l};
  }
}

// fp16 output of DPC dims per query row (8, 16 or 32 bytes) at byte offset off.
template <int DPC>
__device__ __forceinline__ void store_f16_run(__amdgpu_buffer_rsrc_t o_rsrc, uint32_t off, const float* v) {
#pragma unroll
  for (int h8 = 0; h8 < (DPC + 7) / 8; ++h8) {
    constexpr int W = DPC < 8 ? DPC : 8;
    float vals[8];
#pragma unroll
    for (int k8 = 0; k8 < 8; ++k8) vals[k8] = k8 < W ? v[h8 * 8 + (k8 < W ? k8 : 0)] : 0.0f;
    const u32x4 pk = pack_f16x8(vals);
    if constexpr (W == 8) {
      buffer_store16(o_rsrc, off + h8 * 16, pk);
    } else {
      __builtin_amdgcn_raw_buffer_store_b64(u32x2{pk[0], pk[1]}, o_rsrc, (int)off, 0, kPolicyStreamStore);
    }
  }
}

// fp16 output of P.V column n's DPC dims of one query row (dims out_dim(n,
// 0..DPC-1)) whose first element is at byte offset row_off: one contiguous
// run over the row's 16 lanes per store instruction.
template <int DPC>
__device__ __forceinline__ void store_f16_cols(__amdgpu_buffer_rsrc_t o_rsrc, uint32_t row_off, int n,
                                               const float* v) {
  if constexpr (DPC <= 8) {
    store_f16_run<DPC>(o_rsrc, row_off + (uint32_t)out_dim<DPC>(n, 0) * 2u, v);
  } else {
#pragma unroll
    for (int h8 = 0; h8 < DPC / 8; ++h8)
      store_f16_run<8>(o_rsrc, row_off + (uint32_t)out_dim<DPC>(n, 8 * h8) * 2u, v + 8 * h8);
  }
}


// ---------------------------------------------------------------------------
// Single pass on the matrix cores: one (batch, KV head) per workgroup of NW
// waves, all of its query heads in one 16-column tile (G <= 16), K and V
// read once and nothing else in memory.
// ---------------------------------------------------------------------------
// Rows a wave takes (a multiple of the HPW 16-row blocks one round stages),
// for a row bound of nblk 16-row blocks split over NW waves.
template <int D>
constexpr int onepass_mfma_wave_rows(int nblk, int nw) {
  constexpr int RR = GroupShape<D>::HPW * kSplitBlockRows;
  return ((nblk * kSplitBlockRows + nw * RR - 1) / (nw * RR)) * RR;
}
// LDS bytes of one workgroup: the row's fp32 scores ([G][rows + 4], the
// stride off the bank period), the waves' (max, sum) per query column, and
// per wave the K rows / V transpose staging of the matrix-core passes.
template <int D>
constexpr size_t onepass_mfma_lds_bytes(int g, int nblk, int nw) {
  return (size_t)g * (nw * onepass_mfma_wave_rows<D>(nblk, nw) + 4) * 4 + (size_t)nw * 16 * 2 * 4 +
         (size_t)nw * GroupShape<D>::KV_LDS;
}

// Wave w scores rows [w R, w R + R) of the row (R = onepass_mfma_wave_rows)
// a round of HPW 16-row blocks at a time, as the split scores pass does (K
// rows staged in LDS, S^T = K_blk . Q^T on v_mfma_f32_16x16x32_bf16), into
// the workgroup's LDS, keeping per query column a running max and sum of
// exponentials; the next round's K rows are in flight during a round's
// products.  The waves exchange their (max, sum) per column and combine
// them in wave order; each wave then walks V over its rows as the split
// P.V pass does (V^T staged in LDS with v_perm, bf16(exp(t - max) / sum)
// weights as the A operand of v_mfma_f32_16x16x16_bf16), and waves 1..NW-1
// hand their sums to wave 0 through their own staging, which adds them in
// wave order and writes fp16 O.  Packed and strided layouts.
template <int D, int NW, int LAYOUT>
__global__ __launch_bounds__(kBlockThreads * NW) void onepass_mfma_kernel(SplitArgs a) {
  static_assert(LAYOUT == kLayoutPacked || LAYOUT == kLayoutStrided || LAYOUT == kLayoutPagedBlock,
                "packed, strided or pages of at least 16 rows");
  // Paged caches: every lane addresses its own rows (GroupRows), a row in
  // an unmapped page (a negative entry) is read as Q's first row and sets
  // the lane's flag; the (batch, KV head)'s outputs are then NaN.
  constexpr bool PAGED = is_paged_layout(LAYOUT);
  using Sh = GroupShape<D>;
  constexpr int LPH = Sh::LPH;
  constexpr int HPW = Sh::HPW;
  constexpr int NR = kSplitBlockRows;
  constexpr int DPC = Sh::DPC;
  constexpr int RR = HPW * NR;  // rows per round
  extern __shared__ __attribute__((aligned(16))) char onepass_mfma_lds[];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWaveSize));
  const uint32_t hkv = (uint32_t)a.num_heads_kv;
  const uint32_t b = blockIdx.x / hkv;
  const uint32_t hk = blockIdx.x - b * hkv;
  if (b >= (uint32_t)a.batch) return;
  const int hq = a.num_heads_q;
  const int G = hq / (int)hkv;  // <= 16
  const int S = split_len_l<LAYOUT>(a, b);
  const int q = lane >> 4;   // MFMA lane group
  const int n = lane & 15;   // MFMA row / column: this lane's query column
  const int s = lane / LPH;  // load lane group: block s of each round
  const int r = lane % LPH;
  const bool gok = n < G;
  const __amdgpu_buffer_rsrc_t o_rsrc =
      make_rsrc(a.o + ((uint64_t)b * hq + (uint64_t)hk * G) * D, (uint32_t)G * D * 2u);
  if (S <= 0 || S > a.max_rows) {
    // Empty rows give 0 (the reference loop's result), invalid ones NaN.
    if (wv != 0) return;
    const u32x4 fill = S == 0 ? u32x4{0u, 0u, 0u, 0u} : u32x4{0x7e007e00u, 0x7e007e00u, 0x7e007e00u, 0x7e007e00u};
    for (int k = lane; k < G * (D / 8); k += kWaveSize)
      buffer_store16(o_rsrc, (uint32_t)((k / (D / 8)) * D + (k % (D / 8)) * 8) * 2u, fill);
    return;
  }
  const int wrows = onepass_mfma_wave_rows<D>(a.nblk, NW);
  const int sps = NW * wrows + 4;  // floats per query column
  float* sc = reinterpret_cast<float*>(onepass_mfma_lds);
  float* pst = sc + (size_t)G * sps;  // [NW][16][2]
  char* stage = reinterpret_cast<char*>(pst + NW * 16 * 2) + (size_t)wv * Sh::KV_LDS;
  const int lo = wv * wrows;  // this wave's first row
  const int span = S - lo < 0 ? 0 : (S - lo < wrows ? S - lo : wrows);
  const int rounds = (span + RR - 1) / RR;

  // ---- K: scores of rows [lo, lo + span) -> sc, running (max, sum) ----
  GroupRows<D, LAYOUT> kv;
  kv.init(a, a.k, b, split_row_base<LAYOUT>(a, b), 0, S, (int)hk, true, r, s * NR);
  const __amdgpu_buffer_rsrc_t q_rsrc =
      make_rsrc(a.q + ((uint64_t)b * hq + (uint64_t)hk * G) * D, (uint32_t)G * D * 2u);
  bf16x8_v qb[Sh::QLD];
#pragma unroll
  for (int cc = 0; cc < Sh::QLD; ++cc)
    qb[cc] = __builtin_bit_cast(
        bf16x8_v, buffer_load16<kPolicyDefault>(q_rsrc, gok ? (uint32_t)(n * D + (4 * cc + q) * 8) * 2u : kLaneOutOfRange));
  u32x4 kr[NR];
  kv.template load<NR>(kr, lo);
  float rm = -__builtin_inff(), rl = 0.0f;  // this lane's rows of column n
  for (int k = 0; k < rounds; ++k) {
    const int j0 = lo + k * RR;
    wave_lds_sync();  // the previous round's reads of the staging are done
#pragma unroll
    for (int j = 0; j < NR; ++j) *reinterpret_cast<u32x4*>(stage + j * Sh::KS + s * D * 2 + r * 16) = kr[j];
    wave_lds_sync();
    __builtin_amdgcn_sched_barrier(0);
    // The next round's rows are in flight during this round's products
    // (past the wave's rows: rows read 0 without access, or another wave's
    // rows, never used).
    if (k + 1 < rounds) kv.template load<NR>(kr, j0 + RR);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 0; p < HPW; ++p) {
      const int jb = j0 + p * NR;
      if (jb >= lo + span) break;
      f32x4_v c4 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int cc = 0; cc < Sh::QLD; ++cc) {
        const bf16x8_v ka = *reinterpret_cast<const bf16x8_v*>(stage + n * Sh::KS + p * D * 2 + (4 * cc + q) * 16);
        c4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, qb[cc], c4, 0, 0, 0);
      }
      float x[4];
      float bm = -__builtin_inff();
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = c4[e] * a.scale;
        bm = jb + 4 * q + e < S ? fmaxf(bm, x[e]) : bm;
      }
      if (gok)
        *reinterpret_cast<float4*>(sc + (size_t)n * sps + jb + 4 * q) = float4{x[0], x[1], x[2], x[3]};
      const float mn = fmaxf(rm, bm);
      float bs = 0.0f;
#pragma unroll
      for (int e = 0; e < 4; ++e) bs += jb + 4 * q + e < S ? expf(x[e] - mn) : 0.0f;
      rl = rl * (rm == mn ? 1.0f : expf(rm - mn)) + bs;
      rm = mn;
    }
  }
  // The wave's (max, sum) per column: over its four lane groups, then
  // through LDS over the waves, in wave order.
  {
    const float cm = column_reduce<true>(rm);
    const float cl = column_reduce<false>(rl * (rm == cm ? 1.0f : expf(rm - cm)));
    if (q == 0) {
      pst[(wv * 16 + n) * 2] = cm;
      pst[(wv * 16 + n) * 2 + 1] = cl;
    }
  }
  // V rows of the wave's first round, in flight across the exchange.
  GroupRows<D, LAYOUT> vrows;
  vrows.init(a, a.v, b, split_row_base<LAYOUT>(a, b), 0, S, (int)hk, true, r, s * NR);
  u32x4 vr[NR];
  vrows.template load<NR>(vr, lo);
  // Paged: K met an unmapped page among the rows of some wave (V reads the
  // same rows through the same table).
  int poisoned = 0;
  if constexpr (PAGED)
    poisoned = __syncthreads_or(kv.bad != 0);
  else
    __syncthreads();
  float gm = -__builtin_inff();
#pragma unroll
  for (int w = 0; w < NW; ++w) gm = fmaxf(gm, pst[(w * 16 + n) * 2]);
  float gl = 0.0f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float m = pst[(w * 16 + n) * 2];
    gl += m == -__builtin_inff() ? 0.0f : pst[(w * 16 + n) * 2 + 1] * (m == gm ? 1.0f : expf(m - gm));
  }

  // ---- V: rows [lo, lo + span), weights from sc ----
  f32x4_v acc[DPC];
#pragma unroll
  for (int dt = 0; dt < DPC; ++dt) acc[dt] = f32x4_v{0.0f, 0.0f, 0.0f, 0.0f};
  for (int k = 0; k < rounds; ++k) {
    const int j0 = lo + k * RR;
    wave_lds_sync();  // the previous round's reads of the staging are done
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        u32x4 wv4;
#pragma unroll
        for (int pp = 0; pp < 4; ++pp) {
          const int j = 8 * half + 2 * pp;
          wv4[pp] = __builtin_amdgcn_perm((uint32_t)vr[j + 1][e / 2], (uint32_t)vr[j][e / 2],
                                          (e & 1) ? kPermHi : kPermLo);
        }
        *reinterpret_cast<u32x4*>(stage + s * Sh::VSTREAM + r * Sh::VB + e * (NR * 2) + half * 16) = wv4;
      }
    }
    wave_lds_sync();
    if (k + 1 < rounds) vrows.template load<NR>(vr, j0 + RR);
#pragma unroll
    for (int p = 0; p < HPW; ++p) {
      const int jb = j0 + p * NR;
      if (jb >= lo + span) break;
      const char* vs = stage + p * Sh::VSTREAM;
      bf16x4_v vb[DPC];
#pragma unroll
      for (int dt = 0; dt < DPC; ++dt) {
        const int dim = out_dim<DPC>(n, dt);
        vb[dt] = *reinterpret_cast<const bf16x4_v*>(vs + (dim / 8) * Sh::VB + (dim % 8) * (NR * 2) + q * 8);
      }
      const float4 t4 = gok ? *reinterpret_cast<const float4*>(sc + (size_t)n * sps + jb + 4 * q)
                            : float4{0.0f, 0.0f, 0.0f, 0.0f};
      const float tt[4] = {t4.x, t4.y, t4.z, t4.w};
      bf16x4_v pa;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool valid = gok && jb + 4 * q + e < S;
        pa[e] = (__bf16)(valid ? expf(tt[e] - gm) / gl : 0.0f);
      }
#pragma unroll
      for (int dt = 0; dt < DPC; ++dt)
        acc[dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(pa, vb[dt], acc[dt], 0, 0, 0);
    }
  }

  // ---- waves 1..NW-1 -> wave 0 (each through its own staging) ----
  if constexpr (NW > 1) {
    wave_lds_sync();
    if (wv > 0) {
#pragma unroll
      for (int dt = 0; dt < DPC; ++dt)
        *reinterpret_cast<f32x4_v*>(stage + ((size_t)dt * kWaveSize + lane) * 16) = acc[dt];
    }
    __syncthreads();
    if (wv > 0) return;
    for (int w = 1; w < NW; ++w) {
      const char* ws = reinterpret_cast<char*>(pst + NW * 16 * 2) + (size_t)w * Sh::KV_LDS;
#pragma unroll
      for (int dt = 0; dt < DPC; ++dt) {
        const f32x4_v x = *reinterpret_cast<const f32x4_v*>(ws + ((size_t)dt * kWaveSize + lane) * 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[dt][e] += x[e];
      }
    }
  }
  // Lane (q, n) holds query rows 4q..4q+3, dims out_dim(n, 0..DPC-1).
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int g = 4 * q + e;
    float v[DPC];
#pragma unroll
    for (int dt = 0; dt < DPC; ++dt) v[dt] = poisoned ? __builtin_nanf("") : acc[dt][e];
    store_f16_cols<DPC>(o_rsrc, g < G ? (uint32_t)(g * D) * 2u : kLaneOutOfRange, n, v);
  }
}


// ---------------------------------------------------------------------------
// Single pass on the matrix cores, the row's scores in registers.
// ---------------------------------------------------------------------------
// The v_mfma_f32_16x16x32_bf16 scores of a 16-row tile leave lane (q, n)
// (q = lane / 16, n = lane % 16) holding rows 4q..4q+3 of query column n:
// exactly its A operand of v_mfma_f32_16x16x16_bf16 in the P.V product
// (query row n, reduction index 4q + e).  So a wave that keeps its tiles'
// scores in registers needs no LDS for them, and more waves fit a CU than
// with the row's scores in LDS.  Wave w of a workgroup of NW takes rows
// [w R, w R + R), R = 16 TPW, of one (batch, KV head):
//   * K a round of HPW tiles at a time, whole rows per lane group (16 bytes
//     a lane) into a 16-row staging in LDS, read back in the A operand's
//     layout (row n, 16-byte chunks 4c + q; Q's B operand takes the same
//     chunks), the next round's rows in flight during a round's products
//     (loading the A layout straight from memory, 64 bytes of 16 rows per
//     instruction, measured 5-15% slower);
//   * its (max, sum of exp(t - max)) per query column over its rows, those
//     of the workgroup's waves exchanged through LDS and combined in wave
//     order;
//   * V rows 4q..4q+3 of each tile at dims [n D/16, n D/16 + D/16) straight
//     from memory (each load a whole row across the 16 lanes of a lane
//     group), PF tiles in flight, transposed in registers with v_perm into
//     the B operand; weights bf16(exp(t - max) / sum) with the row's global
//     max and sum;
//   * waves 1..NW-1 hand their fp32 sums to wave 0 through LDS (the K
//     staging's space), which adds them in wave order and writes fp16 O.
// Rows past the wave's range are never read (out-of-range offsets read 0).
// A row's tiles are shared evenly among the waves whatever its length, and
// with many workgroups the longest rows go first (longest_of_group): on ragged
// batches a launch otherwise ends on one wave of a late long row (µs, 16-row
// pages, B=64 32/8, lengths log-uniform over 128-4096, 305 MB: 117.6 with
// shares of the longest row in batch order, 69.7; packed B=256 64/8 32-1024:
// 92.4 / 68.6; equal lengths are unchanged, B=256 S=1024 64/8 174.7 / 174.6).
// The tile loops are unrolled over TPW, left at the round after the wave's
// last tile and with no other branch inside: the scores' registers need
// static indices, and a branch per tile made the compiler wait for every
// load in flight at each tile.  Packed and strided layouts,
// and paged ones: pages of at least 16 rows (kLayoutPagedBlock), where a
// tile lies in one page, K through per-lane page addresses (PagedLaneRows),
// V through a descriptor per tile from the tile's block-table entry, which
// each wave requests for all its tiles at the start; smaller pages
// (kLayoutPaged), every row through its own entry and a per-lane address,
// the entries requested ahead of their rows.  A negative entry among a
// (batch, KV head)'s rows makes its outputs NaN, its rows never read.
template <int D, int TPW>
constexpr int onepass_reg_pf() {
  return D == 256 || TPW >= 32 ? 2 : 4;  // V tiles in flight per wave
}
// Tiles per K staging round: a wave's lane groups (HPW) at D >= 128; at
// D = 64 with up to 16 tiles per wave (three or more waves per SIMD by
// registers), and on pages under 16 rows, half of them, two lane groups
// loading 8 rows each of one tile, which halves the staging (more waves
// per CU).
constexpr int onepass_reg_round_tiles(int d, int tpw, int layout) {
  return d == 64 && (tpw <= 16 || layout == kLayoutPaged) ? kWaveSize / (d / 8) / 2 : kWaveSize / (d / 8);
}
// LDS bytes per staged row: the round's tiles' D dims, plus padding.
constexpr int onepass_reg_stage_row(int d, int tpw, int layout) {
  return onepass_reg_round_tiles(d, tpw, layout) * d * 2 + 16;
}
// LDS of a workgroup of nw waves: the (max, sum) exchange, then each wave's
// K staging (16 rows of a round's tiles), whose space the fp32 sums of
// waves 1..nw-1 reuse once every wave is past the exchange.
template <int D>
constexpr size_t onepass_reg_stage_offset(int nw) {
  return (size_t)nw * 16 * 2 * 4;
}
template <int D>
constexpr size_t onepass_reg_lds_bytes(int nw, int tpw, int layout) {
  const size_t stage = (size_t)nw * onepass_reg_stage_row(D, tpw, layout) * kSplitBlockRows;
  const size_t red = (size_t)(nw - 1) * (D / 16) * kWaveSize * 16;
  return onepass_reg_stage_offset<D>(nw) + (stage > red ? stage : red);
}

template <int D, int TPW, int NWMAX, int LAYOUT>
__global__ __launch_bounds__(kBlockThreads * NWMAX) void onepass_mfma_reg_kernel(SplitArgs a) {
  static_assert(LAYOUT == kLayoutPacked || LAYOUT == kLayoutStrided || LAYOUT == kLayoutPagedBlock ||
                    LAYOUT == kLayoutPaged,
                "packed, strided or paged");
  constexpr bool PAGED = LAYOUT == kLayoutPagedBlock;  // pages of at least 16 rows
  constexpr bool PAGED_ROWS = LAYOUT == kLayoutPaged;  // pages under 16 rows
  constexpr int QLD = D / 32;  // 16-byte K chunks per lane per tile
  constexpr int DPC = D / 16;  // output dims per lane (one P.V MFMA each)
  constexpr int VW = DPC / 2;  // dwords of a lane's V run per row
  constexpr int PF = onepass_reg_pf<D, TPW>();
  constexpr int NR = kSplitBlockRows;
  using Sh = GroupShape<D>;
  constexpr int LPH = Sh::LPH;
  constexpr int HPW = Sh::HPW;
  constexpr int RT = onepass_reg_round_tiles(D, TPW, LAYOUT);  // tiles per staging round
  constexpr int KR = NR * RT / HPW;                            // rows a lane group loads per round
  constexpr int KSR = onepass_reg_stage_row(D, TPW, LAYOUT);   // staging bytes per row
  static_assert(TPW % RT == 0, "whole rounds");
  // A wave leaves the tile loops at the round after its last tile, but where
  // running 8 tiles through costs less than the exits (µs with / without:
  // BHSD B=100 S=512 16/16 72.9 / 69.8; packed B=512 S=512 64/8 176.7 /
  // 179.3, ragged B=256 over 16-500 rows 44.6 / 48.0).
  constexpr bool EXITS = TPW > 8 || LAYOUT != kLayoutStrided;
  extern __shared__ __attribute__((aligned(16))) char onepass_reg_lds[];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int nw = (int)(blockDim.x / kWaveSize);
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWaveSize));
  const uint32_t hkv = (uint32_t)a.num_heads_kv;
  const uint32_t bi = blockIdx.x / hkv;
  const uint32_t hk = blockIdx.x - bi * hkv;
  if (bi >= (uint32_t)a.batch) return;
  uint32_t b = bi;
  int S;
  int64_t row_base;
  if (TPW > 8 && __builtin_expect(a.order_groups != 0, 0)) {
    b = longest_of_group<LAYOUT>(a, bi, lane, S, row_base);
  } else {
    S = split_len_l<LAYOUT>(a, b);
    row_base = split_row_base<LAYOUT>(a, b);
  }
  const int hq = a.num_heads_q;
  const int G = hq / (int)hkv;  // <= 16
  const int q = lane >> 4;
  const int n = lane & 15;
  const bool gok = n < G;
  const __amdgpu_buffer_rsrc_t o_rsrc =
      make_rsrc(a.o + ((uint64_t)b * hq + (uint64_t)hk * G) * D, (uint32_t)G * D * 2u);
  if (S <= 0 || S > a.max_rows) {
    // Empty rows give 0 (the reference loop's result), invalid ones NaN.
    if (wv != 0) return;
    const u32x4 fill = S == 0 ? u32x4{0u, 0u, 0u, 0u} : u32x4{0x7e007e00u, 0x7e007e00u, 0x7e007e00u, 0x7e007e00u};
    for (int k = lane; k < G * (D / 8); k += kWaveSize)
      buffer_store16(o_rsrc, (uint32_t)((k / (D / 8)) * D + (k % (D / 8)) * 8) * 2u, fill);
    return;
  }
  // The row's tiles in even shares of whole staging rounds, at most TPW each
  // (a row shorter than the call's longest still keeps every wave busy).
  const uint32_t round_tiles = (uint32_t)(nw * RT);
  const int share = (int)((((uint32_t)(S + NR - 1) / NR + round_tiles - 1) * a.round_inv) >> 16) * RT;
  const int lo = wv * share * NR;
  const int span = S - lo < 0 ? 0 : (S - lo < share * NR ? S - lo : share * NR);
  const int nt = (span + NR - 1) / NR;
  // Pages of at least 16 rows: a tile lies in one page.  Lane t < nt holds
  // the block-table entry of the wave's tile t (entry 0, which a batch with
  // rows always has, elsewhere), requested here, long before V needs it; K
  // and V share the table, so a negative entry among them makes the
  // (batch, KV head) invalid: its outputs are NaN and the unmapped rows are
  // never read.
  int32_t tile_entry = 0;
  int unmapped = 0;
  if constexpr (PAGED) {
    const int32_t* pages = a.block_table + (uint64_t)b * (uint64_t)a.bt_stride;
    const bool has = lane < nt;
    tile_entry = pages[has ? (uint32_t)(lo + lane * NR) >> (uint32_t)a.page_shift : 0u];
    unmapped = __builtin_amdgcn_ballot_w64(has && tile_entry < 0) != 0 ? 1 : 0;
  }

  // ---- K: scores of the wave's tiles, kept in x ----
  // A round of RT tiles: lane group s loads KR rows of tile s % RT (16
  // bytes per lane, chunk r; the whole tile with RT = HPW, its rows 8 (s /
  // RT) on with RT = HPW / 2), stores them to the wave's staging, and the
  // MFMA A operands (row n, chunks 4c + q) are read back from there; the
  // next round's rows are in flight during a round's products.  Tiles past
  // the wave's rows read 0 (without memory access; on pages under 16 rows
  // from Q's first row) and are masked; the loops carry no branch, one
  // branch skips them for a wave without rows.
  const __amdgpu_buffer_rsrc_t q_rsrc =
      make_rsrc(a.q + ((uint64_t)b * hq + (uint64_t)hk * G) * D, (uint32_t)G * D * 2u);
  bf16x8_v qb[QLD];
#pragma unroll
  for (int c = 0; c < QLD; ++c)
    qb[c] = __builtin_bit_cast(
        bf16x8_v, buffer_load16<kPolicyDefault>(q_rsrc, gok ? (uint32_t)(n * D + (4 * c + q) * 8) * 2u : kLaneOutOfRange));
  const int s = lane / LPH;
  const int r = lane % LPH;
  const int ps = s % RT;        // this lane group's tile of a round
  const int ph = (s / RT) * KR;  // and its first row in it
  char* stage = onepass_reg_lds + onepass_reg_stage_offset<D>(nw) + (size_t)wv * KSR * NR;
  typename std::conditional<PAGED || PAGED_ROWS, PagedLaneRows<D, PAGED>, LongRows<D, LAYOUT>>::type kr;
  kr.init(a, a.k, b, row_base, lo, lo + span, (int)hk, true, r, ps * NR + ph);
  f32x4_v x[TPW];
  float m = -__builtin_inff();
  if (nt > 0) {
    u32x4 kb[KR];
    // Pages under 16 rows: each row's block-table entry, requested a round
    // ahead of its rows (entries and rows complete in request order, so
    // the entries of round k + 2 go out after the rows of round k + 1,
    // and waiting for them waits for nothing the round does not need).
    int32_t ek[PAGED_ROWS ? KR : 1];
    if constexpr (PAGED_ROWS) {
      kr.template entries<KR>(ek, 0);
      kr.template load_entries<KR>(kb, 0, ek);
      if (TPW / RT > 1) kr.template entries<KR>(ek, RT * NR);
    } else {
      kr.template load<KR>(kb, 0);
    }
#pragma unroll
    for (int k = 0; k < TPW / RT; ++k) {
      if (EXITS && k * RT >= nt) break;
      wave_lds_sync();  // the previous round's reads of the staging are done
#pragma unroll
      for (int j = 0; j < KR; ++j) *reinterpret_cast<u32x4*>(stage + (ph + j) * KSR + ps * D * 2 + r * 16) = kb[j];
      wave_lds_sync();
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (PAGED_ROWS) {
        if (k + 1 < TPW / RT) {
          kr.template load_entries<KR>(kb, (k + 1) * RT * NR, ek);
          if (k + 2 < TPW / RT) kr.template entries<KR>(ek, (k + 2) * RT * NR);
        }
      } else if (k + 1 < TPW / RT) {
        kr.template load<KR>(kb, (k + 1) * RT * NR);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int p = 0; p < RT; ++p) {
        const int t = k * RT + p;
        f32x4_v c4 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < QLD; ++c) {
          const bf16x8_v ka = *reinterpret_cast<const bf16x8_v*>(stage + n * KSR + p * D * 2 + (4 * c + q) * 16);
          c4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, qb[c], c4, 0, 0, 0);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[t][e] = c4[e] * a.scale;
          m = t * NR + 4 * q + e < span ? fmaxf(m, x[t][e]) : m;
        }
      }
    }
  } else {
#pragma unroll
    for (int t = 0; t < TPW; ++t) x[t] = f32x4_v{0.0f, 0.0f, 0.0f, 0.0f};
  }
  // The wave's (max, sum) per column, over its four lane groups.
  const float cm = column_reduce<true>(m);
  float l = 0.0f;
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
    if (EXITS && t % RT == 0 && t >= nt) break;
#pragma unroll
    for (int e = 0; e < 4; ++e) l += t * NR + 4 * q + e < span ? expf(x[t][e] - cm) : 0.0f;
  }
  const float cl = column_reduce<false>(l);
  float* pst = reinterpret_cast<float*>(onepass_reg_lds);  // [nw][16][2]
  if (q == 0) {
    pst[(wv * 16 + n) * 2] = cm;
    pst[(wv * 16 + n) * 2 + 1] = cl;
  }
  // V rows of the wave's first tiles, in flight across the exchange.
  // A wave of pages under 16 rows has met an unmapped page among its rows
  // if its K loads have (V reads the same rows through the same table).
  if constexpr (PAGED_ROWS) unmapped = __builtin_amdgcn_ballot_w64(kr.bad != 0) != 0 ? 1 : 0;
  LongRows<D, PAGED || PAGED_ROWS ? kLayoutPacked : LAYOUT> vrw;
  if constexpr (!PAGED && !PAGED_ROWS) vrw.init(a, a.v, b, row_base, 0, S, (int)hk, true, 0);
  const uint32_t v_row_bytes = (uint32_t)kv_heads_mem(a) * D * 2u;       // paged: bytes per slot
  const uint32_t v_head_off = (uint32_t)kv_head_mem(a, (int)hk) * D * 2u;  // paged: this KV head in a slot
  uint32_t vr[PF][4][VW];
  // Pages under 16 rows: the entries of this lane's four rows of a tile,
  // requested PF tiles ahead of the tile's rows (after the rows of the tile
  // PF steps earlier, so waiting for them waits only for rows already due).
  int32_t ev[PAGED_ROWS ? PF : 1][4];
  const int32_t* v_pages = a.block_table + (uint64_t)b * (uint64_t)a.bt_stride;
  auto v_entries = [&](int p, int t) {
    if constexpr (PAGED_ROWS) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = t * NR + 4 * q + e;
        ev[p][e] = v_pages[row < span ? (uint32_t)(lo + row) >> (uint32_t)a.page_shift : 0u];
      }
    }
  };
  auto v_load = [&](int p, int t) {
    if constexpr (PAGED_ROWS) {
      // Per-lane addresses; a row past the wave's rows or in an unmapped
      // page reads Q's first row (memory that exists) and becomes 0.
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = t * NR + 4 * q + e;
        const PagedRowU32 pr = paged_row_u32(ev[p][e], (uint32_t)(lo + row), (uint32_t)a.page_shift);
        const bool ok = row < span && !pr.unmapped;
        const uint16_t* src = ok ? a.v + (uint64_t)pr.page * (uint64_t)a.batch_stride +
                                       (uint64_t)pr.slot * (v_row_bytes >> 1) + (v_head_off >> 1) + n * DPC
                                 : a.q;
        if constexpr (VW == 2) {
          const u32x2 w2 = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(src));
          vr[p][e][0] = ok ? w2[0] : 0u;
          vr[p][e][1] = ok ? w2[1] : 0u;
        } else {
#pragma unroll
          for (int h = 0; h < VW / 4; ++h) {
            const u32x4 w4 = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src) + h);
#pragma unroll
            for (int i = 0; i < 4; ++i) vr[p][e][4 * h + i] = ok ? w4[i] : 0u;
          }
        }
      }
      return;
    }
    // Paged: the tile's page through its entry (readlane: no table round
    // trip here), a descriptor over the tile's rows in it (none when the
    // entry is unmapped: nothing is read).
    __amdgpu_buffer_rsrc_t v_rsrc;
    if constexpr (PAGED) {
      const int32_t e = __builtin_amdgcn_readlane(tile_entry, t);
      const PagedRowU32 pr = paged_row_u32(e, (uint32_t)(lo + t * NR), (uint32_t)a.page_shift);
      const int rows = pr.unmapped ? 0 : (span - t * NR < 0 ? 0 : (span - t * NR < NR ? span - t * NR : NR));
      v_rsrc = make_rsrc(uniform_ptr(a.v + (uint64_t)pr.page * (uint64_t)a.batch_stride +
                                     (uint64_t)pr.slot * (v_row_bytes >> 1)),
                         (uint32_t)rows * v_row_bytes);
    } else {
      v_rsrc = vrw.rsrc;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = t * NR + 4 * q + e;
      uint32_t off;
      if constexpr (PAGED)  // from the tile's first row
        off = row < span ? v_head_off + (uint32_t)(4 * q + e) * v_row_bytes + (uint32_t)(n * DPC * 2) : kRowOutOfRange;
      else
        off = row < span ? vrw.lane_off + (uint32_t)(lo + row) * vrw.row_bytes + (uint32_t)(n * DPC * 2)
                         : kRowOutOfRange;
      if constexpr (VW == 2) {
        const u32x2 w2 = __builtin_bit_cast(
            u32x2, __builtin_amdgcn_raw_buffer_load_b64(v_rsrc, (int)off, 0, kPolicyStream));
        vr[p][e][0] = w2[0];
        vr[p][e][1] = w2[1];
      } else {
#pragma unroll
        for (int h = 0; h < VW / 4; ++h) {
          const u32x4 w4 = buffer_load16_nt(v_rsrc, off + (uint32_t)h * 16u);
#pragma unroll
          for (int i = 0; i < 4; ++i) vr[p][e][4 * h + i] = w4[i];
        }
      }
    }
  };
  if constexpr (PAGED_ROWS) {
#pragma unroll
    for (int p = 0; p < PF; ++p) v_entries(p, p);
  }
#pragma unroll
  for (int p = 0; p < PF; ++p) v_load(p, p);
  if constexpr (PAGED_ROWS) {
#pragma unroll
    for (int p = 0; p < PF; ++p) v_entries(p, p + PF);
  }
  const int poisoned = PAGED || PAGED_ROWS ? __syncthreads_or(unmapped) : (__syncthreads(), 0);
  float gm = -__builtin_inff();
  for (int w = 0; w < nw; ++w) gm = fmaxf(gm, pst[(w * 16 + n) * 2]);
  float gl = 0.0f;
  for (int w = 0; w < nw; ++w) {
    const float mw = pst[(w * 16 + n) * 2];
    gl += mw == -__builtin_inff() ? 0.0f : pst[(w * 16 + n) * 2 + 1] * (mw == gm ? 1.0f : expf(mw - gm));
  }

  // ---- V: weights from x ----
  f32x4_v acc[DPC];
#pragma unroll
  for (int dt = 0; dt < DPC; ++dt) acc[dt] = f32x4_v{0.0f, 0.0f, 0.0f, 0.0f};
  if (nt > 0) {
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      if (EXITS && t % RT == 0 && t >= nt) break;
      bf16x4_v pa;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool valid = gok && t * NR + 4 * q + e < span;
        pa[e] = (__bf16)(valid ? expf(x[t][e] - gm) / gl : 0.0f);
      }
      const int p = t % PF;
#pragma unroll
      for (int dt = 0; dt < DPC; ++dt) {
        const uint32_t sel = (dt & 1) ? kPermHi : kPermLo;
        const u32x2 w2 = {__builtin_amdgcn_perm(vr[p][1][dt / 2], vr[p][0][dt / 2], sel),
                          __builtin_amdgcn_perm(vr[p][3][dt / 2], vr[p][2][dt / 2], sel)};
        acc[dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(pa, __builtin_bit_cast(bf16x4_v, w2), acc[dt], 0, 0, 0);
      }
      if (t + PF < TPW) {
        v_load(p, t + PF);
        if (t + 2 * PF < TPW) v_entries(p, t + 2 * PF);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // ---- waves 1..nw-1 -> wave 0 ----
  if (nw > 1) {
    f32x4_v* red = reinterpret_cast<f32x4_v*>(onepass_reg_lds + onepass_reg_stage_offset<D>(nw));
    if (wv > 0) {
#pragma unroll
      for (int dt = 0; dt < DPC; ++dt) red[((size_t)(wv - 1) * DPC + dt) * kWaveSize + lane] = acc[dt];
    }
    __syncthreads();
    if (wv > 0) return;
    for (int w = 1; w < nw; ++w) {
#pragma unroll
      for (int dt = 0; dt < DPC; ++dt) {
        const f32x4_v y = red[((size_t)(w - 1) * DPC + dt) * kWaveSize + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[dt][e] += y[e];
      }
    }
  }
  // Lane (q, n) holds query rows 4q..4q+3, dims [n DPC, n DPC + DPC);
  // NaN for a (batch, KV head) that met an unmapped page.
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int g = 4 * q + e;
    float v[DPC];
#pragma unroll
    for (int dt = 0; dt < DPC; ++dt) v[dt] = poisoned ? __builtin_nanf("") : acc[dt][e];
    store_f16_run<DPC>(o_rsrc, g < G ? (uint32_t)(g * D + n * DPC) * 2u : kLaneOutOfRange, v);
  }
}

}  // namespace fmha_decode
