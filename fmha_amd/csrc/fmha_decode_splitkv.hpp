// fmha_decode_splitkv.hpp -- decode attention for KV lengths beyond 16
// (split-KV), gfx950.
//
// Same semantics as the short-KV kernel, extended to any length S: fp32
// scores, max-subtracted softmax, weights rounded to bf16 *after*
// normalisation (as the reference's CPU loop does, fmha_host.cpp:209-226),
// fp32 P.V, one fp16 rounding.  Because the bf16 rounding needs the global
// max and sum before any weight is formed, the work runs in two launches
// over a caller-provided workspace:
//
//   1. scores (this file; groups of 8 and more on the matrix cores in
//      fmha_decode_splitkv_group.hpp): workgroups of a few waves, one wave
//      per block of 16 rows and KV-head group: the block's Q and K rows are
//      requested at once (as in the short kernel), dot products, transposing
//      butterfly (shared with the short kernel); scaled scores t_j -> T, and
//      per query head the max m and the sum of exp(t_j - m) of the
//      workgroup's rows, joined through LDS.
//   2. P.V (fmha_decode_splitkv_pv.hpp): workgroups of four waves, each
//      joining its row's statistics, weighting a piece of the V rows and, with
//      more than one workgroup per row, leaving a partial output; the last
//      one of a row to finish adds them.
//
// The statistics and the partial outputs once had launches of their own;
// four launches cost a short row more than its bytes (µs of kernels, B=1
// S=3001 32/8 on 16-row pages 20.9 -> 14.1, B=8 of 47-1500 rows 16/16 D=64
// BHSD 17.0 -> 11.8, ragged B=48 8/1 over 250-8000 rows 34.6 -> 24; long rows
// keep their time, B=1 S=131072 104.6 -> 102.0, or gain with groups of 8,
// B=8 S=32768 64/8 221 -> 207).  P.V workgroups find their batch in the
// lengths (row_piece), so that those past the rows of a ragged batch come
// last and end at once, where a grid over the longest row interleaves them
// with the others (µs, B=6 64/8 over 1024-32768 rows on 16-row pages 80.1 /
// 62.9; 84 with four launches); the scores launch's waves are too short for
// the extra round trip (B=8 S=32768 32/8 92 / 97).
//
// K and V are each read once; T adds 4 bytes per row and query head (written
// by 1, read by 2), the statistics 8 bytes per workgroup of 1 and query head
// and the partial outputs 4*D bytes per workgroup of 2 and query head.
#pragma once

#include <type_traits>

#include "fmha_decode_kernel.hpp"
#include "fmha_decode_pieces.hpp"

namespace fmha_decode {

// How a batch's length is found (SplitArgs::len_mode).
constexpr int kLenCu = 0;       // cu[b + 1] - cu[b] (packed layout)
constexpr int kLenArray = 1;    // cu[b] holds the length itself
constexpr int kLenUniform = 2;  // every batch has max_rows rows

typedef float f32x2_v __attribute__((ext_vector_type(2)));

// P.V workgroups of a row whose partial outputs one of them adds.
constexpr int kPvFan = 16;

struct SplitArgs {
  const uint16_t* q;      // [batch, Hq, D] bf16
  const uint16_t* k;      // bf16 K rows in the launch's layout (LongRows)
  const uint16_t* v;
  uint16_t* o;            // [batch, Hq, D] fp16
  const int32_t* cu;      // packed: [batch+1] row offsets; else [batch] lengths (or null, uniform)
  float* t;               // [batch, nblk, Hq, 16] scaled scores
  f32x2_v* st;            // [batch, Hq, nsup] max and sum of exp(t - max) of nsup-th parts of a row
  float* opart;           // [P.V pieces, Hkv, G, D] partial outputs
  uint32_t* done;         // [batch, Hkv, tiles, pv.parts, 1 + ceil(pv.npv / kPvFan)] finished P.V workgroups
  int32_t num_heads_q;
  int32_t num_heads_kv;
  int32_t units_per_batch;  // KV-head groups per batch: ceil(Hkv / HPW)
  int32_t nblk;           // 16-row blocks per batch row: ceil(max_rows / 16)
  PvPieces pv;            // pieces of the P.V launch
  int32_t sup_shift;      // log2 of the rows of a scores workgroup
  int32_t nsup;           // scores workgroups per batch row: ceil(max_rows / 2^sup_shift)
  int32_t max_rows;       // lengths above this are invalid (NaN output)
  int32_t batch;
  float scale;
  int32_t len_mode;       // kLenCu, kLenArray or kLenUniform
  // kLayoutStrided: element strides of K/V; kLayoutPaged: page stride in
  // batch_stride, row (slot) stride in row_stride, block table and
  // log2(page_size).
  int64_t batch_stride;
  int32_t row_stride;
  int32_t head_stride;
  const int32_t* block_table;
  int32_t bt_stride;
  int32_t page_shift;
  // log2 of the sub-units per wave (scores, single pass): with fewer KV
  // heads than a wave holds, its lane groups take 2^sub_shift blocks
  // (scores) of the same heads, or batches (single pass), instead of idling.
  int32_t sub_shift;
  // Launch KV heads per KV head in memory (>= 1): a query group larger than
  // the kernels' G runs as kv_groups groups of G on one launch, launch head
  // hk reading memory head hk / kv_groups of num_heads_kv / kv_groups.
  int32_t kv_groups;
  // Register single pass: ceil(2^16 / n) for the n tiles that the
  // workgroup's waves stage in one round, so that x / n is x * round_inv >>
  // 16 (exact for x * n < 2^16; x is below 512 and n at most 64).
  uint32_t round_inv;
  // Single passes: ceil(batch / 64) with the batches taken about longest row
  // first (longest_of_group), 0: as they come.
  uint32_t order_groups;
};

// KV heads of the cache in memory, and the one launch head hk reads.
__host__ __device__ __forceinline__ int kv_heads_mem(const SplitArgs& a) { return a.num_heads_kv / a.kv_groups; }
__device__ __forceinline__ int kv_head_mem(const SplitArgs& a, int hk) {
  return a.kv_groups == 1 ? hk : hk / a.kv_groups;
}

// Lane groups of a wave under SplitArgs::sub_shift: group hkl (of HPW)
// serves KV head hg * (HPW >> sub_shift) + hkl % (HPW >> sub_shift) for
// sub-unit hkl / (HPW >> sub_shift).
template <int HPW>
struct SubUnits {
  int shift;  // log2(heads per sub-unit)
  __device__ __forceinline__ explicit SubUnits(int sub_shift) : shift(ilog2(HPW) - sub_shift) {}
  __device__ __forceinline__ int heads() const { return 1 << shift; }
  __device__ __forceinline__ int unit(int hkl) const { return hkl >> shift; }
  __device__ __forceinline__ int head(uint32_t hg, int hkl) const { return (int)(hg << shift) + (hkl & (heads() - 1)); }
};

// Length of batch b (may be out of [0, max_rows]: the kernels check).
__device__ __forceinline__ int split_len(const SplitArgs& a, uint64_t b) {
  if (a.len_mode == kLenCu) return a.cu[b + 1] - a.cu[b];
  if (a.len_mode == kLenArray) return a.cu[b];
  return a.max_rows;
}
template <int LAYOUT>
__device__ __forceinline__ int split_len_l(const SplitArgs& a, uint64_t b) {
  if constexpr (LAYOUT == kLayoutPacked) return a.cu[b + 1] - a.cu[b];
  return split_len(a, b);
}

constexpr int kSplitBlockRows = kMaxSeq;  // rows per scores wave

// The lengths of all of a call's batches (at most kOrderBatches), batch p *
// kWaveSize + lane in len[p]; 0 past the last.  Every load is requested at
// once, with no branch between them.
constexpr int kOrderRegs = kOrderBatches / kWaveSize;

template <int LAYOUT>
__device__ __forceinline__ void batch_lengths(const SplitArgs& a, int lane, int (&len)[kOrderRegs]) {
#pragma unroll
  for (int p = 0; p < kOrderRegs; ++p)
    len[p] = split_len_l<LAYOUT>(a, (uint64_t)min(p * kWaveSize + lane, a.batch - 1));
#pragma unroll
  for (int p = 0; p < kOrderRegs; ++p)
    if (p * kWaveSize + lane >= a.batch) len[p] = 0;
}

// The batch that workgroup group i (< batch) of a single-pass launch serves
// with SplitArgs::order_groups (n): about the one with the i-th longest row,
// in 16-row blocks, so that the longest rows start first and the launch does
// not end on one of them alone.  The batches form n strided groups of up to
// 64 (group g: g, g + n, g + 2n, ...), one length per lane, each a sample of
// the whole: every group's longest row goes first, then every group's second
// longest, and so on (exactly in order up to 64 batches).  Group i of the
// launch serves the (i / n)-th longest of group i % n, ties in batch order (a
// group has ceil((batch - g) / n) members, so every batch is served once);
// equal rows come out as they come.  Every lane of the wave calls it; every
// wave of every workgroup finds the same order.  Also gives the length and,
// for packed caches, the batch's first row, which the lanes hold already.
template <int LAYOUT>
__device__ __forceinline__ uint32_t longest_of_group(const SplitArgs& a, uint32_t i, int lane, int& S,
                                                     int64_t& row_base) {
  const uint32_t n = a.order_groups;
  const uint32_t rank = i / n;
  const uint32_t mine = i - rank * n + n * (uint32_t)lane;
  const uint32_t b = min(mine, (uint32_t)a.batch - 1);
  const int first = LAYOUT == kLayoutPacked ? a.cu[b] : 0;
  const int len = LAYOUT == kLayoutPacked ? a.cu[b + 1] - first : split_len_l<LAYOUT>(a, b);
  const int blocks = mine >= (uint32_t)a.batch       ? -1
                     : len < 0 || len > a.max_rows ? 0
                                                   : (len + kSplitBlockRows - 1) / kSplitBlockRows;
  auto at_least = [&](int v) { return __popcll(__builtin_amdgcn_ballot_w64(blocks >= v)); };
  int v = 0;
  for (int bit = 31 - __clz(a.nblk); bit >= 0; --bit)
    if (at_least(v | (1 << bit)) > (int)rank) v |= 1 << bit;
  const int r = (int)rank - at_least(v + 1);  // its place among the rows of v blocks
  const uint64_t m = __builtin_amdgcn_ballot_w64(blocks == v);
  const int before = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
  const int found = (int)__builtin_ctzll(__builtin_amdgcn_ballot_w64(blocks == v && before == r));
  S = __builtin_amdgcn_readlane(len, found);
  row_base = __builtin_amdgcn_readlane(first, found);
  return (uint32_t)__builtin_amdgcn_readlane((int)mine, found);
}

// Wave barrier between LDS writes and reads of one wave.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// What a workgroup of the split passes serves.
struct RowPiece {
  uint32_t b;      // batch
  uint32_t piece;  // rows [piece << shift, (piece + 1) << shift) of it
  int S;           // its length (maybe invalid)
  int shift;
};

// Piece u of a call with `pieces` (those of the longest row) for each batch;
// false for a batch's unused ones, but its first.
template <int LAYOUT>
__device__ __forceinline__ bool batch_piece(const SplitArgs& a, uint32_t u, int shift, uint32_t pieces, RowPiece& out) {
  out.b = u / pieces;
  if (out.b >= (uint32_t)a.batch) return false;
  out.piece = u - out.b * pieces;
  out.S = split_len_l<LAYOUT>(a, out.b);
  out.shift = shift;
  return out.piece == 0 || (out.S <= a.max_rows && (int)(out.piece << shift) < out.S);
}

// Sums of x over lanes 0 .. this one.
__device__ __forceinline__ int wave_scan(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);   // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);   // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);   // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);   // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return x;
}

// The P.V workgroups' pieces: piece u of a call whose batches have
// pv_row_pieces each, in batch order; false past the last.  Up to
// kOrderBatches batches the wave adds up the lengths, so that the workgroups
// past the rows that exist are the last of the grid, and takes shorter pieces
// than the host, which saw only the longest row allowed, where they would
// leave CUs without one (pv_device_shift; µs, B=30 8/8 over 140-4500 rows 45.3
// with the host's 2048 rows, 37.1 with the 1024 taken); above, and with one
// length for all, as batch_piece.  Every lane of every wave of a workgroup
// calls it.
template <int LAYOUT>
__device__ __forceinline__ bool row_piece(const SplitArgs& a, uint32_t u, int lane, RowPiece& out) {
  if (a.len_mode == kLenUniform || a.batch > kOrderBatches)
    return batch_piece<LAYOUT>(a, u, a.pv.shift, (uint32_t)pv_row_pieces(a.max_rows, a.max_rows, a.pv.shift), out);
  if (a.batch == 1) {
    out.b = 0;
    out.piece = u;
    out.S = split_len_l<LAYOUT>(a, 0);
    out.shift = pv_device_shift(a.pv, pv_counted_rows(out.S, a.max_rows));
    return u < (uint32_t)pv_row_pieces(out.S, a.max_rows, out.shift);
  }
  int len[kOrderRegs];
  batch_lengths<LAYOUT>(a, lane, len);
  int rows = 0;
#pragma unroll
  for (int p = 0; p < kOrderRegs; ++p) rows += pv_counted_rows(len[p], a.max_rows);
  out.shift = pv_device_shift(a.pv, __builtin_amdgcn_readlane(wave_scan(rows), kWaveSize - 1));
  uint32_t before = 0;  // pieces of the batches of earlier p
#pragma unroll
  for (int p = 0; p < kOrderRegs; ++p) {
    if (p * kWaveSize >= a.batch) break;
    const int x =
        wave_scan(p * kWaveSize + lane >= a.batch ? 0 : pv_row_pieces(len[p], a.max_rows, out.shift));
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane(x, kWaveSize - 1);
    if (u < before + total) {
      const int l = __popcll(__builtin_amdgcn_ballot_w64(before + (uint32_t)x <= u));
      out.b = (uint32_t)(p * kWaveSize + l);
      out.piece = u - before - (l > 0 ? (uint32_t)__builtin_amdgcn_readlane(x, l - 1) : 0u);
      out.S = __builtin_amdgcn_readlane(len[p], l);
      return true;
    }
    before += total;
  }
  return false;
}

// Joins (max, sum of exp(t - max)) of two parts of a row.  A part without
// rows is (-inf, 0); a NaN sum (an unmapped page, a NaN score) stays NaN.
__device__ __forceinline__ void join_stats(float& m, float& l, float m2, float l2) {
  const float mx = fmaxf(m, m2);
  const float e1 = m == mx ? 1.0f : expf(m - mx);
  const float e2 = m2 == mx ? 1.0f : expf(m2 - mx);
  l = l * e1 + l2 * e2;
  m = mx;
}

__device__ __forceinline__ u32x4 buffer_load16_nt(__amdgpu_buffer_rsrc_t r, uint32_t voffset) {
  return buffer_load16<kPolicyStream>(r, voffset);
}

__device__ __forceinline__ float buffer_load_f32(__amdgpu_buffer_rsrc_t r, uint32_t voffset) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)voffset, 0, kPolicyDefault));
}


// A pointer the whole wave holds, moved to scalar registers: a buffer
// descriptor built from a value the compiler keeps in vector registers
// becomes a loop over the lanes.
__device__ __forceinline__ const uint16_t* uniform_ptr(const uint16_t* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
  return reinterpret_cast<const uint16_t*>(((uint64_t)hi << 32) | lo);
}

// One wave's view of the K (or V) rows [lo, hi) of batch b, in one of the
// layouts of the short kernel:
//   kLayoutPacked:  rows cu[b] + j of [rows, Hkv, D];
//   kLayoutStrided: element b*batch_stride + j*row_stride + h*head_stride + d;
//   kLayoutPaged, kLayoutPagedBlock: slot j % page_size of page
//                   block_table[b][j / page_size] in a [pages, page_size,
//                   Hkv, D] cache.
// load<NR>(out, rel0) fetches rows lo + rel0 .. lo + rel0 + NR - 1 (rel0 a
// multiple of NR, lo a multiple of 16, NR <= 16): 16 bytes per lane, this
// lane's head and dims; rows at or past hi read 0 without memory access, so
// padding, neighbouring batches and unused pages are never read.
template <int D, int LAYOUT>
struct LongRows {
  static constexpr bool PAGED = LAYOUT == kLayoutPaged || LAYOUT == kLayoutPagedBlock;
  __amdgpu_buffer_rsrc_t rsrc;  // packed, strided: rows [lo, hi)
  const uint16_t* base;         // paged: the cache
  const int32_t* pages;         // paged: this batch's block-table row
  uint32_t row_bytes;           // bytes between consecutive rows (slots)
  uint32_t lane_off;            // this lane's head and dims within a row
  int lane_rows;                // rows from lo to this lane's first row (packed, strided)
  int lane_n;                   // rows from lo at which this lane's rows end (packed, strided)
  uint32_t page_shift;
  uint64_t page_stride;         // elements
  int lo, n;                    // first row, rows in range
  // Paged layouts: set once a load has met an unmapped page (a negative
  // block-table entry) among the rows in range; those rows read 0, and the
  // caller makes the batch's outputs NaN (it is invalid).  Wave-uniform: a
  // flag instead of NaN rows keeps the loads free of per-element selects
  // (which took the single pass from 206-221 to 376-382 VGPRs).
  int bad = 0;
  __device__ __forceinline__ bool any_bad() const { return bad != 0; }

  // lane_rows_: this lane's rows start that many rows after lo (lane groups
  // serving different blocks; 0 for the paged layouts).
  __device__ __forceinline__ void init(const SplitArgs& a, const uint16_t* t, uint32_t b, int64_t row_base, int lo_,
                                       int hi, int hk, bool head_ok, int r, int lane_rows_ = 0) {
    lo = lo_;
    n = hi > lo_ ? hi - lo_ : 0;
    lane_rows = lane_rows_;
    lane_n = n;
    const int hkv = kv_heads_mem(a);
    const int hm = kv_head_mem(a, hk);
    if constexpr (LAYOUT == kLayoutPacked) {
      row_bytes = (uint32_t)hkv * D * 2u;
      lane_off = head_ok ? (uint32_t)(hm * D + r * 8) * 2u : kLaneOutOfRange;
      rsrc = make_rsrc(uniform_ptr(t + ((uint64_t)row_base + lo) * hkv * D),
                       (uint32_t)__builtin_amdgcn_readfirstlane(n * (int)row_bytes));
    } else if constexpr (LAYOUT == kLayoutStrided) {
      row_bytes = (uint32_t)a.row_stride * 2u;
      lane_off = head_ok ? (uint32_t)(hm * a.head_stride + r * 8) * 2u : kLaneOutOfRange;
      const uint32_t span = n == 0 ? 0u
                                   : ((uint32_t)(n - 1) * (uint32_t)a.row_stride +
                                      (uint32_t)(hkv - 1) * (uint32_t)a.head_stride + D) * 2u;
      rsrc = make_rsrc(uniform_ptr(t + (uint64_t)b * (uint64_t)a.batch_stride +
                                   (uint64_t)lo * (uint64_t)a.row_stride),
                       (uint32_t)__builtin_amdgcn_readfirstlane((int)span));
    } else {
      row_bytes = (uint32_t)hkv * D * 2u;
      lane_off = head_ok ? (uint32_t)(hm * D + r * 8) * 2u : kLaneOutOfRange;
      base = t;
      pages = a.block_table + (uint64_t)b * (uint64_t)a.bt_stride;
      page_shift = (uint32_t)a.page_shift;
      page_stride = (uint64_t)a.batch_stride;
    }
  }

  // The rows of batches b0 .. b0+nb-1 through one descriptor (packed and
  // strided; lane groups serving different batches): this lane's batch b
  // has S rows (0: nothing is read).  Packed: rows relative to batch b0's
  // first, rel_rows the lane's offset (checked by the caller: rel_rows + S
  // rows stay below 2^30 bytes), the range ending at the last row any lane
  // reads; strided: the nb batches' span with max_rows rows each (checked on
  // the host).  load() then works as for init with lo = 0.
  __device__ __forceinline__ void init_multi(const SplitArgs& a, const uint16_t* t, uint32_t b0, uint32_t nb,
                                             uint32_t b, int S, int rel_rows, int hk, bool head_ok, int r) {
    static_assert(LAYOUT == kLayoutPacked || LAYOUT == kLayoutStrided, "one descriptor per wave");
    lo = 0;
    const int hkv = kv_heads_mem(a);
    const int hm = kv_head_mem(a, hk);
    if constexpr (LAYOUT == kLayoutPacked) {
      row_bytes = (uint32_t)hkv * D * 2u;
      lane_off = head_ok ? (uint32_t)(hm * D + r * 8) * 2u : kLaneOutOfRange;
      lane_rows = rel_rows;
      lane_n = rel_rows + S;
      int m = lane_n;
#pragma unroll
      for (int k = 1; k < kWaveSize; k <<= 1) m = max(m, __shfl_xor(m, k, kWaveSize));
      n = __builtin_amdgcn_readfirstlane(m);
      rsrc = make_rsrc(t + (uint64_t)a.cu[b0] * hkv * D, (uint32_t)n * row_bytes);
    } else {
      row_bytes = (uint32_t)a.row_stride * 2u;
      lane_off = head_ok ? (uint32_t)(hm * a.head_stride + r * 8) * 2u + (b - b0) * (uint32_t)a.batch_stride * 2u
                         : kLaneOutOfRange;
      lane_rows = 0;
      lane_n = S;
      n = a.max_rows;
      const uint32_t span = ((nb - 1) * (uint32_t)a.batch_stride + (uint32_t)(a.max_rows - 1) * (uint32_t)a.row_stride +
                             (uint32_t)(hkv - 1) * (uint32_t)a.head_stride + D) * 2u;
      rsrc = make_rsrc(t + (uint64_t)b0 * (uint64_t)a.batch_stride, span);
    }
  }

  // Descriptor of `rows` rows from row `row` on, inside one page.  A row past
  // the end looks up the entry of a row the wave's range has and gets an
  // empty range.  An unmapped page (a negative block-table entry) gets an
  // empty range too, nothing is read, and `bad` is set when rows > 0.
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t page_rsrc(int row, int rows) {
    const int32_t entry = load_uniform_i32(pages, (uint32_t)row >> page_shift);
    // The scalar unit's form of the guard (a negative entry as page 0 with
    // an empty range).
    const PagedRowU32 pr = paged_row_u32(entry, (uint32_t)row, page_shift);
    bad |= __builtin_amdgcn_readfirstlane(rows > 0 && pr.unmapped ? 1 : 0);
    const uint32_t range = (uint32_t)__builtin_amdgcn_readfirstlane(pr.unmapped ? 0 : rows * (int)row_bytes);
    return make_rsrc(uniform_ptr(base + (uint64_t)pr.page * page_stride + (uint64_t)pr.slot * (row_bytes >> 1)),
                     range);
  }

  template <int NR>
  __device__ __forceinline__ void load(u32x4 (&out)[NR], int rel0) {
    static_assert(NR <= 16, "a sub-block fits a 16-row page");
    if constexpr (LAYOUT == kLayoutPacked || LAYOUT == kLayoutStrided) {
      // Rows past this lane's end are moved out of range (a strided range
      // can also cover other heads' padding rows).  Offsets from one
      // per-lane base plus a wave-uniform step: a per-row multiply of a
      // per-lane row kept 16-32 offsets live (several batches per wave,
      // G = 4: 256 VGPRs and 19 AGPRs against 215; the VALU P.V pass at
      // G = 1: 257 against 169).
      const int rowb = rel0 + lane_rows;
      const uint32_t off0 = lane_off + (uint32_t)rowb * row_bytes;
      const int lim = lane_n - rowb;
#pragma unroll
      for (int j = 0; j < NR; ++j)
        out[j] = buffer_load16_nt(rsrc, j < lim ? off0 + (uint32_t)j * row_bytes : kRowOutOfRange);
    } else if constexpr (LAYOUT == kLayoutPagedBlock) {
      const int valid = n - rel0 < 0 ? 0 : (n - rel0 > NR ? NR : n - rel0);
      const __amdgpu_buffer_rsrc_t pr = page_rsrc(lo + (valid > 0 ? rel0 : 0), valid);
#pragma unroll
      for (int j = 0; j < NR; ++j) out[j] = buffer_load16_nt(pr, lane_off + (uint32_t)j * row_bytes);
    } else {
#pragma unroll
      for (int j = 0; j < NR; ++j) {
        const bool ok = rel0 + j < n;
        out[j] = buffer_load16_nt(page_rsrc(lo + (ok ? rel0 + j : 0), ok ? 1 : 0), lane_off);
      }
    }
  }
};

// The rows [lo, hi) of one (batch, KV head) of a paged cache ([pages,
// page_size, Hkv, D], row j in slot j % page_size of page block_table[b][j /
// page_size]) for waves whose lane groups read different rows: the same
// init / load interface as LongRows, with per-lane addresses.  Each lane
// looks up the pages of its own rows (BLOCK, page_size >= 16: one lookup per
// 16-row block, which lies in one page).  The loads carry no branch (a
// branch in a pipelined loop makes the compiler wait for every request at
// its head): a row at or past the lane's end, or in an unmapped page (a
// negative block-table entry), reads 16 bytes of Q's first row instead --
// memory that always exists -- and is replaced by 0; an unmapped page also
// sets the lane's `bad`, and the caller makes the batch's outputs NaN (an
// invalid batch; a flag rather than NaN rows keeps the loads to one select
// per element: NaN rows took the VALU P.V pass from 245 to 352 VGPRs).
// Block-table lookups stay inside the batch's row (entry 0 for rows past
// the end), and no address is formed from a negative entry.
template <int D, bool BLOCK>
struct PagedLaneRows {
  const uint16_t* base;   // the cache at this lane's head and dims
  const uint16_t* safe;   // 16 readable bytes (Q's first row, this lane's dims)
  const int32_t* pages;   // this batch's block-table row
  uint32_t page_shift;
  uint64_t page_stride;   // elements per page
  uint64_t row_elems;     // elements per slot (Hkv * D)
  int lo, lane_rows, lane_n;
  int bad = 0;  // per lane: a load met an unmapped page among this lane's rows
  // Some lane of the wave met one (the wave's lane groups serve one batch in
  // the split passes).
  __device__ __forceinline__ bool any_bad() const { return __builtin_amdgcn_ballot_w64(bad != 0) != 0; }

  __device__ __forceinline__ void init(const SplitArgs& a, const uint16_t* t, uint32_t b, int64_t, int lo_, int hi,
                                       int hk, bool head_ok, int r, int lane_rows_ = 0) {
    const int n = hi > lo_ ? hi - lo_ : 0;
    lo = lo_;
    lane_rows = lane_rows_;
    lane_n = head_ok ? n : 0;
    base = t + (uint64_t)kv_head_mem(a, hk) * D + r * 8;
    safe = a.q + r * 8;
    pages = a.block_table + (uint64_t)b * (uint64_t)a.bt_stride;
    page_shift = (uint32_t)a.page_shift;
    page_stride = (uint64_t)a.batch_stride;
    row_elems = (uint64_t)kv_heads_mem(a) * D;
  }

  // Rows lo + rel0 + lane_rows + j, j < NR (lo and lane_rows multiples of
  // 16, rel0 a multiple of NR <= 16: with BLOCK the NR rows lie in one
  // 16-row block, hence in one page).  entries() requests their block-table
  // entries (one per row, or one with BLOCK) and load_entries() the rows
  // through them, so that a caller can request the entries a step ahead:
  // the entries and rows are vector loads, which complete in order, so
  // requesting both in one step makes every step wait a table round trip
  // after the previous rows.
  template <int NR>
  static constexpr int kEntries = BLOCK ? 1 : NR;

  template <int NR>
  __device__ __forceinline__ void entries(int32_t (&e)[kEntries<NR>], int rel0) const {
    const int row0 = rel0 + lane_rows;
    if constexpr (BLOCK) {
      const uint32_t abs0 = (uint32_t)(lo + row0);
      e[0] = pages[row0 < lane_n ? abs0 >> page_shift : 0u];
    } else {
#pragma unroll
      for (int j = 0; j < NR; ++j) {
        const uint32_t abs = (uint32_t)(lo + row0 + j);
        e[j] = pages[row0 + j < lane_n ? abs >> page_shift : 0u];
      }
    }
  }

  template <int NR>
  __device__ __forceinline__ void load_entries(u32x4 (&out)[NR], int rel0, const int32_t (&e)[kEntries<NR>]) {
    const int row0 = rel0 + lane_rows;
    u32x4 v[NR];
    bool unmapped[NR];
    // The guard in unsigned factors (paged_row_u32: a negative entry as
    // page 0, never read): the signed 64-bit form cost registers.
    if constexpr (BLOCK) {
      const bool any = row0 < lane_n;
      const PagedRowU32 pr = paged_row_u32(e[0], (uint32_t)(lo + row0), page_shift);
      const uint64_t el = (uint64_t)pr.page * page_stride + (uint64_t)pr.slot * row_elems;
#pragma unroll
      for (int j = 0; j < NR; ++j) {
        const bool ok = !pr.unmapped && row0 + j < lane_n;
        v[j] = __builtin_nontemporal_load(
            reinterpret_cast<const u32x4*>(ok ? base + el + (uint64_t)j * row_elems : safe));
        unmapped[j] = any && pr.unmapped;
      }
    } else {
#pragma unroll
      for (int j = 0; j < NR; ++j) {
        const bool ok = row0 + j < lane_n;
        const PagedRowU32 pr = paged_row_u32(e[j], (uint32_t)(lo + row0 + j), page_shift);
        const uint64_t el = (uint64_t)pr.page * page_stride + (uint64_t)pr.slot * row_elems;
        v[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(ok && !pr.unmapped ? base + el : safe));
        unmapped[j] = ok && pr.unmapped;
      }
    }
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      const bool ok = row0 + j < lane_n && !unmapped[j];
      bad |= unmapped[j] ? 1 : 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) out[j][k] = ok ? (uint32_t)v[j][k] : 0u;
    }
  }

  template <int NR>
  __device__ __forceinline__ void load(u32x4 (&out)[NR], int rel0) {
    int32_t e[kEntries<NR>];
    entries<NR>(e, rel0);
    load_entries<NR>(out, rel0, e);
  }
};

// The row loader of the split-KV passes for a layout.
template <int D, int LAYOUT>
using SplitRows = typename std::conditional<LAYOUT == kLayoutPagedLanes || LAYOUT == kLayoutPagedBlockLanes,
                                            PagedLaneRows<D, LAYOUT == kLayoutPagedBlockLanes>,
                                            LongRows<D, LAYOUT>>::type;

// First packed row of batch b (0 for the other layouts, which address rows
// per batch).
template <int LAYOUT>
__device__ __forceinline__ int64_t split_row_base(const SplitArgs& a, uint64_t b) {
  if constexpr (LAYOUT == kLayoutPacked) return a.cu[b];
  return 0;
}

// ---------------------------------------------------------------------------
// 1. scores
// ---------------------------------------------------------------------------
// Scores of 16-row block blk of batch b live at
// T[((b * nblk + blk) * Hq + query head) * 16 + row % 16]: each wave writes
// one contiguous span (its heads' 16 rows), whole cache lines.
__device__ __forceinline__ uint64_t t_block_base(const SplitArgs& a, uint64_t b, int blk) {
  return ((b * (uint64_t)a.nblk + (uint64_t)blk) * (uint64_t)a.num_heads_q) * kSplitBlockRows;
}

// One 16-row block per lane group, all of its K rows requested at once: a
// wave serves 2^sub_shift consecutive blocks (SubUnits).  The G query heads
// of a KV head are scored GH at a time against the same K registers (GH = 4
// bounds the partial sums a lane holds to 64).  A workgroup's waves take the
// next blocks of the same heads and join their statistics through LDS.
// One wave, but on rows of more than kScoresLongBlocks blocks kScoresMaxWaves
// (half of them with one or two query heads per KV head): more, held until the slowest is done, measured slower (µs of this
// launch at 1 / 2 / 4 / 8 waves, 32/8 D=128: B=1 S=131072 47.9 / 50.8 / 50.4
// / 52.1, S=3001 4.9 / 5.6 / 6.4 / 8.0, B=8 S=32768 92.4 / 97.3), and fewer
// leave the P.V launch more entries to join than its lanes take at once (S =
// 131072 53.9 with four waves here, 56.8 with two; µs of the call at 1 / 2 / 4
// waves, 16/16 B=1 S=60000 87.0 / 84.7 / 89.5, 32/16 88.2 / 86.0 / 91.4, 8/8 D=256
// S=70000 110.9 / 106.2 / 109.1, 32/32 D=64 S=71980 121.4 / 117.0 / 118.8, 32/8 D=64
// S=131072 80.0 / 73.1 / 69.2).  Grid: pieces
// (batch_piece) of 2^sup_shift rows times units_per_batch head groups.
constexpr int kScoresMaxWaves = 4;
constexpr int kScoresLongBlocks = 2048;

// Zeroes the P.V arrival counts of `heads` KV heads from hk0 on of batch b,
// `subs` (query tiles times parts of the dims) each; the workgroups of the P.V
// launch count from it.
__device__ __forceinline__ void clear_done(const SplitArgs& a, uint32_t b, uint32_t hk0, int heads, int subs) {
  if (a.pv.npv == 1) return;
  const uint32_t per = (uint32_t)(subs * (1 + (a.pv.npv + kPvFan - 1) / kPvFan));
  const uint32_t n = min((uint32_t)heads, (uint32_t)a.num_heads_kv - min(hk0, (uint32_t)a.num_heads_kv)) * per;
  uint32_t* done = a.done + ((uint64_t)b * a.num_heads_kv + hk0) * per;
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) done[i] = 0u;
}

template <int D, int G, int LAYOUT = kLayoutPacked>
__global__ __launch_bounds__(kBlockThreads * kScoresMaxWaves) void splitkv_scores_kernel(SplitArgs a) {
  constexpr int LPH = D / 8;
  constexpr int HPW = kWaveSize / LPH;
  constexpr int NS = ilog2(LPH);
  constexpr int NR = kSplitBlockRows;
  constexpr int GH = G > 4 ? 4 : G;
  constexpr int V = GH * NR;
  constexpr int L = NS < ilog2(V) ? NS : ilog2(V);
  constexpr int W = (V >> NS) > 1 ? (V >> NS) : 1;
  constexpr int GS = W < NR ? W : NR;
  constexpr int C = ilog2(NR / GS);
  __shared__ f32x2_v st_lds[kScoresMaxWaves][HPW][G];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWaveSize));
  // Workgroup order (piece, head group): consecutive ones read neighbouring
  // heads of the same rows.
  const SubUnits<HPW> su(a.sub_shift);
  const uint32_t upb = (uint32_t)a.units_per_batch;
  const uint32_t u = blockIdx.x / upb;
  const uint32_t hg = blockIdx.x - u * upb;
  RowPiece rp;
  if (!batch_piece<LAYOUT>(a, u, a.sup_shift, (uint32_t)a.nsup, rp)) return;
  const uint32_t b = rp.b;
  const int S = rp.S;
  // Ahead of clear_done's stores, behind which it is a vector load.
  const int64_t row_base = split_row_base<LAYOUT>(a, b);
  if (rp.piece == 0) clear_done(a, b, hg * su.heads(), su.heads(), a.pv.parts);
  if (S <= 0 || S > a.max_rows) return;
  const uint32_t wb = (rp.piece << (a.sup_shift - a.sub_shift - ilog2(NR))) + (uint32_t)wv;
  const int j0 = (int)(wb << a.sub_shift) * NR;  // the wave's first row
  const int hkl = lane / LPH;
  const int p = su.unit(hkl);           // this lane group's block of the wave
  const int hk = su.head(hg, hkl);
  const bool head_ok = hk < a.num_heads_kv;
  const int r = lane % LPH;
  const int hq = a.num_heads_q;
  const int jb = j0 + p * NR;           // first row of this lane group's block
  const bool block_ok = jb < S;         // else past the row (and maybe past nblk): no writes
  for (int i = lane; i < HPW * G; i += kWaveSize) st_lds[wv][i / G][i % G] = f32x2_v{-__builtin_inff(), 0.0f};
  __builtin_amdgcn_wave_barrier();
  if (j0 < S) {  // wave-uniform
  const __amdgpu_buffer_rsrc_t q_rsrc = make_rsrc(a.q + (uint64_t)b * hq * D, (uint32_t)hq * D * 2);
  // Rows [0, S) of the batch: rows past S read 0 without access.
  SplitRows<D, LAYOUT> kv;
  kv.init(a, a.k, b, row_base, 0, S, hk, head_ok, r, p * NR);
  const uint32_t q_off = head_ok ? (uint32_t)(hk * G * D + r * 8) * 2u : kLaneOutOfRange;

  u32x4 qv[G];
#pragma unroll
  for (int g = 0; g < G; ++g) qv[g] = buffer_load16<kPolicyDefault>(q_rsrc, q_off + g * D * 2);
  u32x4 ks[NR];
  kv.template load<NR>(ks, j0);
  __builtin_amdgcn_sched_barrier(0);
  const bool kv_bad = kv.any_bad();

  // After the butterfly, lane r holds scores [blkl*W, blkl*W + W) of the
  // GH*NR (query head, row) pairs; lanes equal in r >> (NS - L) hold copies.
  const int blkl = r >> (NS - L);
  const bool writer = head_ok && block_ok && (r & ((1 << (NS - L)) - 1)) == 0;
  {
    // The wave's blocks' scores [Hq][16] each, written non-temporally (read
    // once, by the P.V pass): 4-6% faster on long-context shapes than
    // default-policy stores.  The range ends at the batch's last block.
    const int wblk = (int)(wb << a.sub_shift);
    const int nwblk = a.nblk - wblk < (1 << a.sub_shift) ? a.nblk - wblk : (1 << a.sub_shift);
    const __amdgpu_buffer_rsrc_t t_rsrc =
        make_rsrc(a.t + t_block_base(a, b, wblk), (uint32_t)nwblk * (uint32_t)hq * NR * 4u);
    const uint32_t t_lane = head_ok ? ((uint32_t)p * hq + (uint32_t)hk * G) * NR * 4u : kLaneOutOfRange;
#pragma unroll
    for (int g0 = 0; g0 < G; g0 += GH) {
      u32x4 qh[GH];
#pragma unroll
      for (int g = 0; g < GH; ++g) qh[g] = qv[g0 + g];
      float x[V];
      partial_scores<GH, NR>(qh, ks, x);
      TransposeReduce<LPH, V, 0>::run(x, lane);
#pragma unroll
      for (int h = 0; h < W / GS; ++h) {
        float t[GS];
        float bm = -__builtin_inff();
        const int vi0 = blkl * W + h * GS;
        const int g = g0 + vi0 / NR;
        const int jr0 = vi0 % NR;
#pragma unroll
        for (int w = 0; w < GS; ++w) {
          t[w] = x[h * GS + w] * a.scale;
          bm = jb + jr0 + w < S ? fmaxf(bm, t[w]) : bm;
        }
        // Scores of rows past S (their K rows read as 0) land in the
        // block's padding, which nothing reads as a weight.
        if (writer) {
          const uint32_t off = t_lane + (uint32_t)(g * NR + jr0) * 4u;
          if constexpr (GS % 4 == 0) {
#pragma unroll
            for (int w = 0; w < GS; w += 4) {
              const u32x4 v4 = {__builtin_bit_cast(uint32_t, t[w]), __builtin_bit_cast(uint32_t, t[w + 1]),
                                __builtin_bit_cast(uint32_t, t[w + 2]), __builtin_bit_cast(uint32_t, t[w + 3])};
              __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_gcc, v4), t_rsrc, (int)(off + w * 4),
                                                     0, kPolicyStreamStore);
            }
          } else {
#pragma unroll
            for (int w = 0; w < GS; ++w)
              __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, t[w]), t_rsrc, (int)(off + w * 4), 0,
                                                    kPolicyStreamStore);
          }
        }
        // Every block has a valid row, so the group's max is finite for
        // finite scores.
        bm = GroupReduce<LPH, L - C, L, true>::run(bm);
        float bs = 0.0f;
#pragma unroll
        for (int w = 0; w < GS; ++w) bs += jb + jr0 + w < S ? expf(t[w] - bm) : 0.0f;
        bs = GroupReduce<LPH, L - C, L, false>::run(bs);
        if (writer && (blkl & ((1 << C) - 1)) == 0) {
          // An unmapped page among the block's rows: a NaN sum makes every
          // weight of the batch's heads, hence its outputs, NaN.
          st_lds[wv][hkl][g] = f32x2_v{bm, kv_bad ? __builtin_nanf("") : bs};
        }
      }
    }
  }
  }
  __syncthreads();
  // The workgroup's statistics of each query head, waves and lane groups in
  // row order.
  for (int i = (int)threadIdx.x; i < su.heads() * G; i += (int)blockDim.x) {
    const int h = i / G, g = i % G;
    const int hko = su.head(hg, h);
    if (hko >= a.num_heads_kv) continue;
    float m = -__builtin_inff(), l = 0.0f;
    for (int w = 0; w < (int)blockDim.x / kWaveSize; ++w)
      for (int q = 0; q < (1 << a.sub_shift); ++q) {
        const f32x2_v x = st_lds[w][(q << su.shift) + h][g];
        join_stats(m, l, x[0], x[1]);
      }
    a.st[((uint64_t)b * hq + (uint64_t)hko * G + g) * a.nsup + rp.piece] = f32x2_v{m, l};
  }
}

}  // namespace fmha_decode
