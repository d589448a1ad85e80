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

// Workgroups a plan for full rows asks for, about two for each CU, all of them
// at once (µs of the call at 2048 / 4096 rows, 32/8 B=8 S=32768 194.4 / 192.3,
// 64/8 218.6 / 207.0; P.V alone, B=1 S=131072 71 / 59 / 54 at 512 / 1024 /
// 2048).  At 256 dims, with twice the bytes in flight for each wave or head,
// fewer do (8/1 B=9 S=40879 on 64-row pages, by halves, 180 workgroups 82.1,
// 720 85.9; 64/8 B=16 S=4096 256 95.4, 512 100.0; 16/2 B=4 S=16384 on 16-row
// pages 256 37.7, 512 40.1, 128 41.0).
constexpr int64_t kPvMinGroups = 448, kPvMinGroupsWide = 176;
// Ragged batches: the workgroups below which the device takes shorter pieces
// (from pv.big on kPvMinGroups; µs by rows, their workgroups in brackets: B=48
// 8/1 over 250-8000 rows 26.9 (420) / 25.1 (210) / 26.6 (105) at 256 / 512 /
// 1024; B=6 64/8 over 1024-32768 64.9 (430) / 63.3 (215) / 73.4 (107) at 1024
// / 2048 / 4096; D=64 B=22 8/8 over 666-21321 65.3 (512) / 71.5 (256) at 2048
// / 4096; D=256 B=8 40/8 over 188-6000 on 64-row pages 39.7 (425) / 41.3
// (212) at 512 / 1024).
constexpr int64_t kPvFewGroups = 192;

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

// The plan for batch rows of up to max_rows on hkv KV heads: the longest
// pieces that leave enough workgroups, but not a size that leaves the last of
// two or three pieces of a row mostly empty (64-row pages D=64 B=57 8/8 S=2233:
// 67.6 at 2048 rows, 58.1 at 1024, 52.8 in one), and, where the device adds up
// the lengths, no row of more than 1024 in one piece in a ragged batch (packed
// D=64 8/8 over 62-2000 rows: B=120 40.1 in one, 37.9 at 1024, but B=300 75.5
// and 88.5, where the pieces that short rows don't have are launched too).  At 256 dims with fewer than
// kPvMinGroupsWide pieces of kPvMaxShift, two workgroups share a head's dims:
// half the sums for each (µs, one / two: B=1 32/4 S=5000 24.8 / 18.8, 32/1
// S=4000 28.5 / 20.5, 64/8 B=16 S=4096 99.1 / 95.4; above, each reads half of
// every 512 bytes: 28/4 B=3 S=66558 162 / 170, BHSD 32/16 B=1 S=61035 160 /
// 165).  forced_rows > 0: pieces of so many rows, everywhere.
inline PvPieces plan_pv_pieces(int64_t batch, int hkv, int max_rows, int d, int forced_rows) {
  const auto groups = [&](int s) { return max_rows <= 0 ? 1 : ((int64_t)max_rows + (1 << s) - 1) >> s; };
  PvPieces pv{};
  const bool wide = d == 256;
  const int64_t enough = wide ? kPvMinGroupsWide : kPvMinGroups;
  pv.parts = wide && batch * hkv * groups(kPvMaxShift) < enough ? 2 : 1;
  const int64_t heads = (int64_t)hkv * pv.parts;
  const auto fits = [&](int s) {
    const int64_t n = groups(s);
    if (n > 1 && n < 4 && (int64_t)max_rows * 10 < 7 * (n << s)) return false;
    return batch * heads * n >= enough;
  };
  pv.shift = kPvMaxShift;
  while (pv.shift > kPvMinShift && !fits(pv.shift)) --pv.shift;
  if (forced_rows > 0)
    for (pv.shift = 0; 1 << pv.shift < forced_rows;) ++pv.shift;
  pv.fine = forced_rows > 0 || batch > kOrderBatches || pv.shift < kPvMinShift ? pv.shift : kPvMinShift;
  pv.most = pv.shift;
  while (pv.most > pv.fine && max_rows > 1024 && groups(pv.most) == 1) --pv.most;
  pv.few = (int32_t)((kPvFewGroups + heads - 1) / heads);
  pv.many = (int32_t)((kPvMinGroups + heads - 1) / heads);
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
