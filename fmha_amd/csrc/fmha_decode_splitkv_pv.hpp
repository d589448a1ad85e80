// fmha_decode_splitkv_pv.hpp -- the P.V launch of the split-KV passes
// (lengths beyond 16 rows): row statistics, weights, P.V and the sum over a
// row's workgroups, gfx950.
//
// A workgroup of kPvWaves waves takes 2^shift V rows (row_piece) of one (batch, KV
// head) for up to 16 of its query heads (a tile), all of its dims or half of
// them (PARTS = 2); larger groups and halves take several workgroups, placed
// on one XCD so that V or the scores come from its L2 after the first:
//   * its waves request their first scores T and V tiles, then join the
//     statistics that the scores launch left per part of the row into each
//     query head's max and sum;
//   * wave w takes the 16-row tiles w, w + kPvWaves, ... in groups of GT:
//     the group's 16 * GT * GC weights bf16(exp(t - max) / sum), GC >= G
//     query columns, are formed one per lane and step (the matrix cores'
//     own layout would have every lane form 4 per tile, 16 / G times too
//     many) and pass through LDS into the A operand of DV/16 (DV: the
//     workgroup's dims)
//     v_mfma_f32_16x16x16_bf16 per tile; V comes straight from memory in the
//     B operand's rows (lane (q, n): rows 4q..4q+3 at dims [n DV/16,
//     +DV/16)), transposed in registers with v_perm, GT tiles in flight;
//   * the waves' fp32 sums are added in wave order through LDS and written
//     as fp16 O by a row's only workgroup, else as fp32 partial outputs, of
//     which the last workgroup to finish of each kPvFan neighbours adds
//     theirs, and the last of those the sums, in row order.
//
// Finding the last one.  Partial outputs are stored as relaxed agent-scope
// atomics, which write through the XCD's L2; every wave waits for its stores
// (s_waitcnt vmcnt(0)) before the workgroup counts itself with one
// agent-scope atomic add, and the workgroup that finds all others counted
// loads them as relaxed agent-scope atomics, past any stale line.  An
// agent-scope release fence instead would write back the whole L2 (about
// 350 ns each, one after another).  No workgroup ever waits for another.  The
// counts are zeroed by the scores launch.
//
// Four waves per workgroup: with eight, two workgroups per CU start and end
// together, nothing streaming meanwhile (µs of this launch, 32/8 B=1
// S=131072 80 / 65, B=48 8/1 over 250-8000 rows 28 / 16).  What bounds it: V's
// bytes for long rows (5.6 TB/s at B=1 S=131072, 51.5 us; D = 256 28/4 B=3
// S=66558 on 64-row pages 5.0 TB/s, 87.9 us), behind each workgroup's joining of
// the whole row's statistics; for short ones the chain lengths -> scores and V
// -> weights -> sums -> count, about 8 us.  Every descriptor comes from scalar
// registers: from vector ones each load was a loop over the lanes (µs of the
// call, packed MQA 32/1 B=16 S=32768 93.8 / 91.4, 8/8 D = 256 B=10 up to 11516
// rows on 16-row pages 58.5 / 55.9).  The order of every sum is fixed, whichever workgroup is last.
#pragma once

#include "fmha_decode_group.hpp"
#include "fmha_decode_splitkv.hpp"
#include "fmha_decode_splitkv_group.hpp"

namespace fmha_decode {

constexpr int kPvWaves = 4;
constexpr int kPvThreads = kPvWaves * kWaveSize;
// Rows of at most this many: one wave, whose lanes join the statistics of
// all of a tile's query heads at once, four entries each.
constexpr int kPvOneWaveRows = 64;

// Tiles per group: as many V tiles as a wave keeps in flight (four measured
// the same and leave half the waves per SIMD).
constexpr int kPvGroupTiles = 2;

// LDS bytes: the waves' weights of a tile group, then (reusing them) their
// sums.
template <int DV, int GC>
constexpr int pv_lds_bytes() {
  constexpr int weights = kPvWaves * kPvGroupTiles * GC * kSplitBlockRows * 2;
  constexpr int sums = kPvWaves * GC * DV * 4;
  return weights > sums ? weights : sums;
}

// One wave's V tiles (16 rows of one (batch, KV head) each, the workgroup's
// dims) in the B operand's rows: lane (q, n) gets rows 4q..4q+3 at dims
// out_dim(n, 0..DPC-1), so that each load instruction reads whole lines of a
// row (µs of the call at D = 256, 16 neighbouring dims per lane / this: 28/4
// B=3 S=66558 on 64-row pages 197 / 179, packed 64/8 B=16 S=4096 106 / 101).
// Tiles are step_tiles apart from row `first` on; rows at or past
// `end` read 0, without memory access (on pages under 16 rows from Q's first
// row).  Paged: an unmapped page (a negative entry) reads as 0 too; the
// scores launch has made the batch's statistics NaN then.
template <int D, int LAYOUT, int PARTS>
struct VTiles {
  static constexpr bool PAGED = LAYOUT == kLayoutPagedBlock;    // a tile lies in one page
  static constexpr bool PAGED_ROWS = LAYOUT == kLayoutPaged;    // every row through its own entry
  static constexpr int DPC = D / PARTS / 16;
  static constexpr int VW = DPC / 2;              // dwords of a lane's dims of a row
  static constexpr int RUN = out_dim<DPC>(0, 8);  // dims from a lane's first 16 bytes of a row to its next
  __amdgpu_buffer_rsrc_t rsrc;  // packed, strided: the batch's rows
  const uint16_t* v;
  const uint16_t* safe;
  const int32_t* pages;
  uint32_t row_bytes, lane_off, page_shift;
  uint64_t page_stride;
  int first, end, step, q;
  int32_t tile_entry;  // PAGED: lane k holds the entry of the wave's tile k (64 at most)

  __device__ __forceinline__ void init(const SplitArgs& a, uint32_t b, int hk, int part, int S, int first_, int end_,
                                       int step_tiles, int lane) {
    uint32_t head_off;
    first = first_;
    end = end_;
    step = step_tiles * kSplitBlockRows;
    q = lane >> 4;
    if constexpr (PAGED || PAGED_ROWS) {
      v = a.v;
      safe = a.q;
      pages = a.block_table + (uint64_t)b * (uint64_t)a.bt_stride;
      page_shift = (uint32_t)a.page_shift;
      page_stride = (uint64_t)a.batch_stride;
      row_bytes = (uint32_t)kv_heads_mem(a) * D * 2u;
      head_off = (uint32_t)kv_head_mem(a, hk) * D * 2u;
      if constexpr (PAGED) {
        const int row = first + lane * step;
        tile_entry = pages[row < end ? (uint32_t)row >> page_shift : 0u];
      }
    } else {
      LongRows<D, LAYOUT> rows;
      rows.init(a, a.v, b, split_row_base<LAYOUT>(a, b), 0, S, hk, true, 0);
      rsrc = rows.rsrc;
      row_bytes = rows.row_bytes;
      head_off = rows.lane_off;
    }
    lane_off = head_off + (uint32_t)(part * (D / PARTS) + out_dim<DPC>(lane & 15, 0)) * 2u + (PAGED_ROWS ? 0u : 4u * (uint32_t)q * row_bytes);
  }

  // PAGED_ROWS: the block-table entries of this lane's rows of tile k, to be
  // requested a group ahead of the rows (loads complete in order).
  __device__ __forceinline__ void entries(int32_t (&e)[4], int k) const {
    if constexpr (PAGED_ROWS) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = first + k * step + 4 * q + i;
        e[i] = pages[row < end ? (uint32_t)row >> page_shift : 0u];
      }
    }
  }

  __device__ __forceinline__ void load(uint32_t (&out)[4][VW], int k, const int32_t (&entry)[4]) const {
    const int row0 = first + k * step;
    if constexpr (PAGED_ROWS) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = row0 + 4 * q + i;
        const PagedRowU32 pr = paged_row_u32(entry[i], (uint32_t)row, page_shift);
        const bool ok = row < end && !pr.unmapped;
        const uint16_t* src = ok ? v + (uint64_t)pr.page * page_stride + (uint64_t)pr.slot * (row_bytes >> 1) +
                                       (lane_off >> 1)
                                 : safe;
        if constexpr (VW == 2) {
          const u32x2 w = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(src));
          out[i][0] = ok ? w[0] : 0u;
          out[i][1] = ok ? w[1] : 0u;
        } else {
#pragma unroll
          for (int h = 0; h < VW / 4; ++h) {
            const u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src + h * RUN));
#pragma unroll
            for (int j = 0; j < 4; ++j) out[i][4 * h + j] = ok ? w[j] : 0u;
          }
        }
      }
    } else {
      __amdgpu_buffer_rsrc_t r;
      uint32_t at = 0;  // of the tile's first row in the range (a valid row's whole offset is in range)
      if constexpr (PAGED) {
        // One descriptor per tile, over the tile's rows in its page (none
        // when the entry is unmapped).
        const int32_t e = __builtin_amdgcn_readlane(tile_entry, k);
        const PagedRowU32 pr = paged_row_u32(e, (uint32_t)row0, page_shift);
        const int left = end - row0;
        const int rows = pr.unmapped || left < 0 ? 0 : (left < kSplitBlockRows ? left : kSplitBlockRows);
        r = make_rsrc(uniform_ptr(v + (uint64_t)pr.page * page_stride + (uint64_t)pr.slot * (row_bytes >> 1)),
                      (uint32_t)__builtin_amdgcn_readfirstlane(rows * (int)row_bytes));
      } else {
        r = rsrc;
        at = (uint32_t)row0 * row_bytes;
      }
      const int left = end - row0 - 4 * q;  // of this lane's four rows
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int off = (int)(i < left ? lane_off + (uint32_t)i * row_bytes : kRowOutOfRange);
        if constexpr (VW == 2) {
          const u32x2 w =
              __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, off, (int)at, kPolicyStream));
          out[i][0] = w[0];
          out[i][1] = w[1];
        } else {
#pragma unroll
          for (int h = 0; h < VW / 4; ++h) {
            const u32x4 w = __builtin_bit_cast(
                u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off + h * (RUN * 2), (int)at, kPolicyStream));
#pragma unroll
            for (int j = 0; j < 4; ++j) out[i][4 * h + j] = w[j];
          }
        }
      }
    }
  }
};

// Max or sum over the wave's lanes, in a fixed order, in every lane.
template <bool IS_MAX>
__device__ __forceinline__ float wave_total(float x) {
  const auto step = [&](auto from) {
    const float y = __builtin_bit_cast(float, from(__builtin_bit_cast(int, IS_MAX ? x : 0.0f), __builtin_bit_cast(int, x)));
    x = IS_MAX ? fmaxf(x, y) : x + y;
  };
  step([](int old, int v) { return __builtin_amdgcn_update_dpp(old, v, 0x111, 0xf, 0xf, false); });  // row_shr:1
  step([](int old, int v) { return __builtin_amdgcn_update_dpp(old, v, 0x112, 0xf, 0xf, false); });  // row_shr:2
  step([](int old, int v) { return __builtin_amdgcn_update_dpp(old, v, 0x114, 0xf, 0xf, false); });  // row_shr:4
  step([](int old, int v) { return __builtin_amdgcn_update_dpp(old, v, 0x118, 0xf, 0xf, false); });  // row_shr:8
  step([](int old, int v) { return __builtin_amdgcn_update_dpp(old, v, 0x142, 0xa, 0xf, false); });  // row_bcast:15
  step([](int old, int v) { return __builtin_amdgcn_update_dpp(old, v, 0x143, 0xc, 0xf, false); });  // row_bcast:31
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), kWaveSize - 1));
}

// Two neighbouring floats of a partial output, past the XCD's L2.
__device__ __forceinline__ void store_partial(float* p, f32x2_v x) {
  __hip_atomic_store(reinterpret_cast<uint64_t*>(p), __builtin_bit_cast(uint64_t, x), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ f32x2_v load_partial(const float* p) {
  return __builtin_bit_cast(f32x2_v, __hip_atomic_load(reinterpret_cast<const uint64_t*>(p), __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT));
}

// Counts this workgroup's finished stores (every thread's) at *count; true
// in every thread when it is the last of n.
__device__ __forceinline__ bool last_to_finish(uint32_t* count, uint32_t n, uint32_t* flag) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0)
    *flag = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  return __builtin_amdgcn_readfirstlane((int)*flag) == (int)n - 1;
}

// Sum of n partial outputs, `stride` floats apart, in order.
__device__ __forceinline__ f32x2_v sum_partials(const float* p, int n, size_t stride) {
  constexpr int U = 8;
  f32x2_v s = {0.0f, 0.0f};
  for (int c0 = 0; c0 < n; c0 += U) {
    f32x2_v x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = load_partial(p + (size_t)(c0 + u < n ? c0 + u : c0) * stride);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c0 + u < n) s += x[u];
  }
  return s;
}

// Grid: units = pieces (row_piece) * Hkv, unit u * Hkv + hk, each with `subs`
// workgroups: ceil(G / 16) query tiles times PARTS parts of the dims; ceil(units / 8) * 8 * subs workgroups, workgroup w serving
// unit ((w / 8) / subs) * 8 + w % 8 and tile and part (w / 8) % subs, so that
// one unit's run on one XCD (dispatch is round-robin over the 8 XCDs).  GC:
// query columns formed, at least min(G, 16).
template <int D, int GC, int LAYOUT, int PARTS>
__global__ __launch_bounds__(kPvThreads) void splitkv_pv_kernel(SplitArgs a) {
  using VT = VTiles<D, LAYOUT, PARTS>;
  constexpr int NR = kSplitBlockRows;
  constexpr int DPC = VT::DPC;
  constexpr int DV = D / PARTS;  // the workgroup's dims
  constexpr int GT = kPvGroupTiles;
  constexpr int SLOTS = GT * NR * GC;                                 // weights of a tile group
  constexpr int PL = (SLOTS + kWaveSize - 1) / kWaveSize;             // per lane
  constexpr int ND = GC >= 4 ? GC / 4 : 1;                            // query columns a lane's slots cover
  static_assert(GC == 1 || GC == 2 || GC == 4 || GC == 8 || GC == 16, "query columns");
  __shared__ __attribute__((aligned(16))) char lds[pv_lds_bytes<DV, GC>()];
  __shared__ f32x2_v heads[GC];  // (max, sum) per query column
  __shared__ uint32_t flag;
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWaveSize));
  const int nw = (int)(blockDim.x / kWaveSize);  // kPvWaves, or 1 on short rows
  const uint32_t hkv = (uint32_t)a.num_heads_kv;
  const int hq = a.num_heads_q;
  const int G = hq / (int)hkv;
  const uint32_t tiles = (uint32_t)(G + 15) / 16;
  const uint32_t part = (blockIdx.x >> 3) % (uint32_t)PARTS;
  const uint32_t rest = (blockIdx.x >> 3) / (uint32_t)PARTS;
  const uint32_t qt = tiles == 1 ? 0 : rest % tiles;
  const uint32_t unit = (tiles == 1 ? rest : rest / tiles) * 8u + (blockIdx.x & 7u);
  const uint32_t u = unit / hkv;
  const uint32_t hk = unit - u * hkv;
  RowPiece rp;
  if (!row_piece<LAYOUT>(a, u, lane, rp)) return;
  const uint32_t b = rp.b;
  const int S = rp.S;
  const int gn = G - (int)qt * 16 < GC ? G - (int)qt * 16 : GC;  // query heads of this tile
  const uint64_t head0 = (uint64_t)b * hq + (uint64_t)hk * G + qt * 16;
  // The workgroup's dims of its query heads' outputs, D apart.
  const __amdgpu_buffer_rsrc_t o_rsrc = make_rsrc(a.o + head0 * D + part * DV, (uint32_t)((gn - 1) * D + DV) * 2u);
  if (S <= 0 || S > a.max_rows) {
    // Empty rows give 0 (the reference loop's result), invalid ones NaN.
    const u32x4 fill = S == 0 ? u32x4{0u, 0u, 0u, 0u} : u32x4{0x7e007e00u, 0x7e007e00u, 0x7e007e00u, 0x7e007e00u};
    for (int i = (int)threadIdx.x; i < gn * (DV / 8); i += (int)blockDim.x)
      buffer_store16(o_rsrc, (uint32_t)(i / (DV / 8) * D + i % (DV / 8) * 8) * 2u, fill);
    return;
  }
  const int row0 = (int)rp.piece << rp.shift;
  const int end = S - row0 < (1 << rp.shift) ? S : row0 + (1 << rp.shift);
  const int first = row0 + wv * NR;  // the wave's first tile
  const int nt = end <= first ? 0 : (end - first + nw * NR - 1) / (nw * NR);
  const int groups = (nt + GT - 1) / GT;

  // Slot f = lane + 64 i of a group is (tile f / (16 GC), query column (f /
  // 16) % GC, row f % 16), a tile's scores being 16 GC neighbouring floats:
  // tile lane_tile + slot_tile(i), column lane_col + 4 (i % ND).
  const int lane_tile = GC < 4 ? lane / (NR * GC) : 0;
  const int lane_col = (lane / NR) % (GC < 4 ? GC : 4);
  const auto slot_tile = [](int i) { return GC < 4 ? i * (4 / GC) : i / (GC < 4 ? 1 : GC / 4); };
  const int lane_row = lane_tile * nw * NR + lane % NR;
  bool col_ok[ND];
#pragma unroll
  for (int i = 0; i < ND; ++i) col_ok[i] = lane_col + 4 * i < gn;
  const __amdgpu_buffer_rsrc_t t_rsrc =
      make_rsrc(a.t + t_block_base(a, b, 0), (uint32_t)a.nblk * (uint32_t)hq * NR * 4u);
  const uint32_t t_tile = (uint32_t)(nw * NR * 4) * (uint32_t)hq;  // bytes from a tile to the wave's next
  const uint32_t t_off = ((uint32_t)(first / NR + lane_tile * nw) * hq + hk * G + qt * 16 + lane_col) * (NR * 4) +
                         (uint32_t)(lane % NR) * 4u;
  // Past the row: scores of other columns or rows, or nothing, masked below.
  float t[PL];
  auto load_t = [&](int k) {
#pragma unroll
    for (int i = 0; i < PL; ++i)
      t[i] = buffer_load_f32(t_rsrc,
                             t_off + (uint32_t)(i % ND) * (4 * NR * 4) + (uint32_t)(k * GT + slot_tile(i)) * t_tile);
  };
  VT vt;
  vt.init(a, b, (int)hk, (int)part, S, first, end, nw, lane);
  uint32_t vr[GT][4][VT::VW];
  int32_t ev[GT][4];
  // The row's statistics: wave w joins those of query columns w, w + kPvWaves,
  // ..., SU per lane requested ahead of the scores and V.
  constexpr int HW = (GC + kPvWaves - 1) / kPvWaves;
  constexpr int SU = HW == 1 ? 32 : HW == 2 ? 16 : 8;
  const int ns = (S + (1 << a.sup_shift) - 1) >> a.sup_shift;
  const __amdgpu_buffer_rsrc_t st_rsrc = make_rsrc(a.st + head0 * a.nsup, (uint32_t)gn * (uint32_t)a.nsup * 8u);
  constexpr int SF = 4;  // short rows have no more
  const bool few = ns <= SF * kWaveSize;
  f32x2_v st[HW][SU];
  auto load_st = [&](f32x2_v (&x)[SU], int h, int s0) {
#pragma unroll
    for (int i = 0; i < SU; ++i) {
      if (i == SF && few) break;
      const int s = s0 + i * kWaveSize + lane;
      const uint32_t off = s < ns ? (uint32_t)((wv + h * kPvWaves) * a.nsup + s) * 8u : kLaneOutOfRange;
      x[i] = __builtin_bit_cast(f32x2_v, __builtin_amdgcn_raw_buffer_load_b64(st_rsrc, (int)off, 0, kPolicyDefault));
    }
  };
  auto join_lane = [&](float& m, float& l, const f32x2_v (&x)[SU], int s0) {
    float mx = m;
#pragma unroll
    for (int i = 0; i < SU; ++i) {
      if (i == SF && few) break;
      mx = s0 + i * kWaveSize + lane < ns ? fmaxf(mx, x[i][0]) : mx;
    }
    l *= m == mx ? 1.0f : expf(m - mx);
#pragma unroll
    for (int i = 0; i < SU; ++i) {
      if (i == SF && few) break;
      const float y = x[i][1] * (x[i][0] == mx ? 1.0f : expf(x[i][0] - mx));
      l += s0 + i * kWaveSize + lane < ns ? y : 0.0f;
    }
    m = mx;
  };
  f32x2_v one = {-__builtin_inff(), 0.0f};  // one wave: entry lane % 4 of column lane / 4
  if (nw == 1) {
    if (lane / 4 < gn && lane % 4 < ns) one = a.st[(head0 + lane / 4) * a.nsup + lane % 4];
  } else {
#pragma unroll
    for (int h = 0; h < HW; ++h) load_st(st[h], h, 0);
  }
  load_t(0);
#pragma unroll
  for (int p = 0; p < GT; ++p) vt.entries(ev[p], p);
#pragma unroll
  for (int p = 0; p < GT; ++p) vt.load(vr[p], p, ev[p]);
#pragma unroll
  for (int p = 0; p < GT; ++p) vt.entries(ev[p], GT + p);

  // Join the row's statistics, those past the first SU per lane after V.
  if (nw == 1) {
    float m = one[0], l = one[1];
#pragma unroll
    for (int d = 1; d < 4; d <<= 1) join_stats(m, l, __shfl_xor(m, d, kWaveSize), __shfl_xor(l, d, kWaveSize));
    if (lane % 4 == 0 && lane / 4 < gn) heads[lane / 4] = f32x2_v{m, l};
  }
#pragma unroll
  for (int h = 0; h < HW; ++h) {
    const int g = wv + h * kPvWaves;
    if (nw == 1 || g >= gn) break;
    float m = -__builtin_inff(), l = 0.0f;
    join_lane(m, l, st[h], 0);
    for (int s0 = SU * kWaveSize; s0 < ns; s0 += SU * kWaveSize) {
      load_st(st[h], h, s0);
      join_lane(m, l, st[h], s0);
    }
    const float mw = wave_total<true>(m);
    l = wave_total<false>(l * (m == mw ? 1.0f : expf(m - mw)));
    m = mw;
    if (lane == 0) heads[g] = f32x2_v{m, l};
  }
  __syncthreads();
  float gm[ND], gl[ND];
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    gm[i] = col_ok[i] ? heads[lane_col + 4 * i][0] : 0.0f;
    gl[i] = col_ok[i] ? heads[lane_col + 4 * i][1] : 1.0f;
  }

  // ---- weights and P.V ----
  const int q = lane >> 4;
  const int n = lane & 15;
  char* w_lds = lds + wv * (SLOTS * 2);
  f32x4_v acc[DPC];
#pragma unroll
  for (int d = 0; d < DPC; ++d) acc[d] = f32x4_v{0.0f, 0.0f, 0.0f, 0.0f};
  for (int k = 0; k < groups; ++k) {
    const int left = end - first - k * (GT * nw * NR);  // rows from the wave's first tile of the group
    uint16_t* w = reinterpret_cast<uint16_t*>(w_lds);
#pragma unroll
    for (int i = 0; i < PL; ++i) {
      const bool ok = col_ok[i % ND] && lane_row + slot_tile(i) * (nw * NR) < left;
      const float p = ok ? expf(t[i] - gm[i % ND]) / gl[i % ND] : 0.0f;
      if (SLOTS >= kWaveSize || lane < SLOTS) w[lane + kWaveSize * i] = __builtin_bit_cast(uint16_t, (__bf16)p);
    }
    load_t(k + 1);
    wave_lds_sync();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 0; p < GT; ++p) {
      // Query column n (columns at or past GC repeat others and are not stored).
      const bf16x4_v pa = *reinterpret_cast<const bf16x4_v*>(w_lds + (p * GC + n % GC) * (NR * 2) + q * 8);
#pragma unroll
      for (int d = 0; d < DPC; ++d) {
        const uint32_t sel = (d & 1) ? kPermHi : kPermLo;
        const u32x2 vb = {__builtin_amdgcn_perm(vr[p][1][d / 2], vr[p][0][d / 2], sel),
                          __builtin_amdgcn_perm(vr[p][3][d / 2], vr[p][2][d / 2], sel)};
        acc[d] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(pa, __builtin_bit_cast(bf16x4_v, vb), acc[d], 0, 0, 0);
      }
      vt.load(vr[p], (k + 1) * GT + p, ev[p]);
      vt.entries(ev[p], (k + 2) * GT + p);
      __builtin_amdgcn_sched_barrier(0);
    }
    wave_lds_sync();  // the weights are read
  }

  // Lane (q, n) holds query columns 4q..4q+3, dims out_dim(n, 0..DPC-1).
  if (nw == 1) {  // the row's only wave
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v[DPC];
#pragma unroll
      for (int d = 0; d < DPC; ++d) v[d] = acc[d][e];
      const int g = 4 * q + e;
      store_f16_cols<DPC>(o_rsrc, g < gn ? (uint32_t)(g * D) * 2u : kLaneOutOfRange, n, v);
    }
    return;
  }

  // ---- the waves' sums, in wave order ----
  __syncthreads();  // the weights are read
  float* red = reinterpret_cast<float*>(lds);  // [wave][GC][DV]
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int g = 4 * q + e;
    if (g < GC) {
#pragma unroll
      for (int d4 = 0; d4 < DPC / 4; ++d4)
        *reinterpret_cast<f32x4_v*>(red + (wv * GC + g) * DV + out_dim<DPC>(n, 4 * d4)) =
            f32x4_v{acc[4 * d4][e], acc[4 * d4 + 1][e], acc[4 * d4 + 2][e], acc[4 * d4 + 3][e]};
    }
  }
  __syncthreads();
  constexpr int PT = (GC * DV / 2 + kPvThreads - 1) / kPvThreads;  // pairs of dims per thread
  const int pairs = gn * (DV / 2);
  f32x2_v sum[PT];
  // Thread t's i-th pair, 2 * (t + i * kPvThreads) floats on.
  auto each = [&](auto body) {
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int e = (int)threadIdx.x + i * kPvThreads;
      if (e < pairs) body(i, 2 * e);
    }
  };
  each([&](int i, int e) {
    sum[i] = f32x2_v{0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < kPvWaves; ++w)
      sum[i] += *reinterpret_cast<const f32x2_v*>(red + w * (GC * DV) + e);
  });

  // ---- a row's workgroups, kPvFan at a time, in row order ----
  const int np = (S + (1 << rp.shift) - 1) >> rp.shift;  // of this row
  if (np > 1) {
    const int nfan = (a.pv.npv + kPvFan - 1) / kPvFan;  // of the longest row
    // Piece c of the row leaves its heads' sums at out + c * stride.
    const size_t stride = (size_t)hq * D;
    float* out = a.opart + (uint64_t)(u - rp.piece) * stride + ((uint64_t)hk * G + qt * 16) * D + part * (gn * DV);
    uint32_t* done = a.done + ((((uint64_t)b * hkv + hk) * tiles + qt) * PARTS + part) * (1 + nfan);
    const int fan = (int)rp.piece / kPvFan;
    const int fan_n = np - fan * kPvFan < kPvFan ? np - fan * kPvFan : kPvFan;
    each([&](int i, int e) { store_partial(out + rp.piece * stride + e, sum[i]); });
    if (!last_to_finish(done + 1 + fan, (uint32_t)fan_n, &flag)) return;
    each([&](int i, int e) { sum[i] = sum_partials(out + (size_t)fan * kPvFan * stride + e, fan_n, stride); });
    if (np > kPvFan) {
      // In the place of the first of them, which this thread has read.
      each([&](int i, int e) { store_partial(out + (size_t)fan * kPvFan * stride + e, sum[i]); });
      const int fans = (np + kPvFan - 1) / kPvFan;
      if (!last_to_finish(done, (uint32_t)fans, &flag)) return;
      each([&](int i, int e) { sum[i] = sum_partials(out + e, fans, kPvFan * stride); });
    }
  }
  each([&](int i, int e) {
    const uint32_t h0 = __builtin_bit_cast(uint16_t, (_Float16)sum[i][0]);
    const uint32_t h1 = __builtin_bit_cast(uint16_t, (_Float16)sum[i][1]);
    __builtin_amdgcn_raw_buffer_store_b32(h0 | (h1 << 16), o_rsrc, (e / DV * D + e % DV) * 2, 0, kPolicyStreamStore);
  });
}

}  // namespace fmha_decode
