// fmha_decode_pieces.hpp -- how the split-KV P.V launch shares out rows: the
// host's plan from what it knows of a call, and the device's choice from the
// lengths.
//
// A workgroup takes a piece of 2^shift rows of one (batch, KV head), all of
// its dims or half of them.  A piece costs about 8 us of start and end however
// short it is (lengths, statistics, sums over waves and workgroups), and
// fewer, longer ones also read memory in fewer places at once; too few leave
// CUs idle.
//
// Plain integer arithmetic, compiled for the device by the kernels and for
// the host by the CPU test (tests/test_pv_pieces.py).
#pragma once

#include <stdint.h>

#include "fmha_decode_paged.hpp"  // FMHA_DECODE_HD

namespace fmha_decode {

constexpr int kPvMinShift = 8, kPvMaxShift = 12;  // planned pieces: 256 to 4096 rows
// Batches up to which the device adds up the lengths.
constexpr int kOrderBatches = 256;

// What of a piece's start and end its CU's other workgroups don't hide, in rows
// of it, and the CUs.
constexpr int64_t kPvPieceRows = 400, kPvSlowPieceRows = 600;
constexpr int kPvCusShift = 8;  // log2
// Pieces of kPvMaxShift from which on a workgroup takes all of 256 dims.
constexpr int64_t kPvWholeGroups = 176;
// Ragged batches: the workgroups below which the device takes shorter pieces,
// and those below which it does from pv.big on; one with a group above 8 counts
// twice (µs by rows, their workgroups in brackets: B=48
// 8/1 over 250-8000 rows 26.9 (420) / 25.1 (210) / 26.6 (105) at 256 / 512 /
// 1024; B=6 64/8 over 1024-32768 64.9 (430) / 63.3 (215) / 73.4 (107) at 1024
// / 2048 / 4096; D=64 B=22 8/8 over 666-21321 65.3 (512) / 71.5 (256) at 2048
// / 4096; D=256 B=8 40/8 over 188-6000 on 64-row pages 39.7 (425) / 41.3
// (212) at 512 / 1024; 32/1 B=48 over 97-3119 28.0 (330) / 25.0 (170) at 256 /
// 512).
constexpr int64_t kPvFewGroups = 192, kPvManyGroups = 448;

struct PvPieces {
  int32_t shift;  // log2 of a piece's rows where the batches are full,
  int32_t most;   // the most where they are not,
  int32_t fine;   // and the least the device may make it
  int32_t few;    // pieces of rows / 2^shift below which it is,
  int32_t many;   // and those below which it is from `big` on
  int32_t big;
  int32_t full;   // rows (pv_counted_rows) from which on the batches are full
  int32_t parts;  // workgroups that share a head's dims
  int32_t npv;    // pieces of a row, at most
  int64_t total;  // pieces of the call, at most
};

// A batch's rows as the device adds them up: 0 where invalid, and capped, so
// that the sum over kOrderBatches stays below 2^31 (a row at the cap alone
// makes more pieces than any plan is short of).
FMHA_DECODE_HD int pv_counted_rows(int S, int max_rows) {
  return S <= 0 || S > max_rows ? 0 : (S < (1 << 22) ? S : 1 << 22);
}

// Pieces of a batch of S rows: one of an empty or invalid batch, which writes
// its output.
FMHA_DECODE_HD int pv_row_pieces(int S, int max_rows, int shift) {
  return S <= 0 || S > max_rows ? 1 : (int)(((uint32_t)S + (1u << shift) - 1) >> shift);
}

// The device's choice, from the sum of pv_counted_rows.
FMHA_DECODE_HD int pv_device_shift(const PvPieces& pv, int rows) {
  if (rows >= pv.full) return pv.shift;
  int s = pv.most;
  while (s > pv.fine && (rows >> s) < (s >= pv.big ? pv.many : pv.few)) --s;
  return s;
}

// The plan for `batch` rows of up to max_rows and `units` (KV head, query tile)
// pairs of groups of g: the size whose busiest CU is done first.  While all workgroups start
// at once (four to a CU, three of 256 dims) that CU has one more of them than
// others may, each as long as a full piece; more of them fill up the CUs as
// they free up.  A CU streams for about one workgroup at a time, whatever it
// holds, but for two where they are slow: at 64 dims, with groups above 8
// (weights of 16 query columns) and on scattered rows (pages under 16 rows, an
// entry for each), and then with no fewer than kPvManyGroups, but for groups
// above 8.  µs of the call by rows, with the workgroups in brackets: 32/32
// D=128 B=9 S=6663 on 16-row pages 186.4 (576) / 168.5 (1152) / 170.3 (2016) at
// 4096 / 2048 / 1024; 32/8 B=1 S=131072 102.2 (256) / 103.4 (512) / 106.9
// (1024); 16/2 D=256 B=4 S=16384 41.1 (128) / 37.9 (256) / 40.5 (512) at 2048 /
// 1024 / 512; 8/8 D=64 B=57 S=2233 on 64-row pages 53.1 (456) / 68.3 (912) / 58.5
// (1368) at 4096 / 2048 / 1024; 4/1 D=64 B=12 S=30000 44.4 (96) / 35.2 (180) /
// 33.1 (360) / 33.4 (708) at 4096 / 2048 / 1024 / 512; 32/1 B=60 S=4777 on 16-row
// pages 74.0 (240) / 68.9 (360) / 64.7 (600) at 4096 / 2048 / 1024; BHSD 28/4 B=23
// S=1208 29.1 (184) / 25.3 (460) at 1024 / 256; one-row pages D=128 32/8 B=1
// S=100000 102.9 (200) / 92.8 (392) / 98.5 (784) at 4096 / 2048 / 1024, 16/16 B=2
// S=9000 47.9 (160) / 42.7 (288) / 40.4 (576) at 2048 / 1024 / 512.
//
// Rows of up to 512 are one piece (µs at 256 / 512 rows, S=300 8/8 D=128 B=4 11.3
// / 10.7, 32/8 B=8 on 16-row pages 13.8 / 12.8; S=512 11.6 / 11.4, 14.1 / 14.1).
// With more batches than the device adds up, the longest of at most 2048 rows
// that leave kPvManyGroups: the pieces that short rows don't have are launched
// too (packed D=64 8/8 B=300 over 62-2000 rows 75.5 in one piece each, 88.5 at
// 1024; 32/1 B=291 over 22-713 29.7 in one, 37.7 at 512; BHSD D=64 4/1 B=764
// over 160-5107 88 at 2048, 107 at 4096).
//
// A ragged batch takes no more than a third of its longest row at once, from
// 1024 rows on (packed D=64 8/8 B=120 over 62-2000 rows 40.1 in one, 37.9 at
// 1024; 16-row pages B=100 over 94-3000 48.1 at 2048, 44.2 at 1024).
//
// At 256 dims with fewer than kPvWholeGroups pieces of kPvMaxShift, two
// workgroups share a head's dims: half the sums for each (µs, one / two: B=1
// 32/4 S=5000 24.8 / 18.8, 32/1 S=4000 28.5 / 20.4, 64/8 B=16 S=4096 99.1 /
// 95.4; above, each reads half of every 512 bytes: 28/4 B=3 S=66558 162 / 170,
// BHSD 32/16 B=1 S=61035 160 / 165).  forced_rows > 0: pieces of so many rows,
// everywhere.
inline PvPieces plan_pv_pieces(int64_t batch, int units, int g, int max_rows, int d, bool scattered,
                               int forced_rows) {
  const auto groups = [&](int s) { return max_rows <= 0 ? 1 : ((int64_t)max_rows + (1 << s) - 1) >> s; };
  PvPieces pv{};
  const bool wide = d == 256;
  pv.parts = wide && batch * units * groups(kPvMaxShift) < kPvWholeGroups ? 2 : 1;
  const int64_t heads = (int64_t)units * pv.parts;
  const bool slow = d == 64 || scattered;
  const int places = kPvCusShift + (slow || g > 8 ? 1 : 0);  // log2
  const int64_t ends = slow ? kPvSlowPieceRows : kPvPieceRows;
  const int64_t at_once = (int64_t)(wide && pv.parts == 1 ? 3 : 4) << kPvCusShift;
  const auto cost = [&](int s) {  // in half rows
    const int64_t n = groups(s), w = batch * heads * n;
    if (w <= at_once) return 2 * ((w + (1 << places) - 1) >> places) * ((n == 1 ? max_rows : 1 << s) + ends);
    return ((2 * w + ((slow ? 2 : 1) << places)) * ((max_rows + n - 1) / n + ends)) >> places;
  };
  const int least = max_rows <= 1 << (kPvMinShift + 1) ? kPvMinShift + 1 : kPvMinShift;
  pv.shift = batch > kOrderBatches ? kPvMaxShift - 1 : kPvMaxShift;
  int64_t best = cost(pv.shift);
  for (int s = pv.shift - 1; s >= least; --s) {
    const bool few = batch * heads * groups(pv.shift) < kPvManyGroups;
    const int64_t c = cost(s);
    if (batch > kOrderBatches ? few : c < best || (slow && few)) {
      pv.shift = s;
      best = c;
    }
  }
  if (forced_rows > 0)
    for (pv.shift = 0; 1 << pv.shift < forced_rows;) ++pv.shift;
  pv.fine = forced_rows > 0 || batch > kOrderBatches || pv.shift < least ? pv.shift : least;
  pv.most = pv.shift;
  while (pv.most > pv.fine && pv.most > 10 && groups(pv.most) < 3) --pv.most;
  const int64_t counted = heads * (g > 8 ? 2 : 1);
  pv.few = (int32_t)((kPvFewGroups + counted - 1) / counted);
  pv.many = (int32_t)((kPvManyGroups + counted - 1) / counted);
  pv.big = wide ? 10 : kPvMaxShift;
  const int64_t allowed = batch * pv_counted_rows(max_rows, max_rows);  // below 2^31 where the device adds up
  pv.full = allowed / 4 * 3 < INT32_MAX ? (int32_t)(allowed / 4 * 3) : INT32_MAX;
  pv.npv = (int32_t)groups(pv.fine);
  // Pieces of 2^most rows, or the shorter ones that the device takes where
  // there are fewer than `many` of twice their rows, and one more per batch.
  const int64_t coarse = batch * groups(pv.most), fine = batch * groups(pv.fine);
  const int64_t few = 2 * (int64_t)(pv.many > pv.few ? pv.many : pv.few) + batch;
  pv.total = coarse > few ? coarse : (fine < few ? fine : few);
  return pv;
}

}  // namespace fmha_decode
