// pv_pieces_shim.cpp -- the split-KV P.V launch's plan of pieces
// (fmha_decode_pieces.hpp, the header the host and the kernels include),
// compiled for the host so that tests/test_pv_pieces.py can drive it on the
// CPU.  Test infrastructure only; the test compiles it with g++ into a
// temporary directory.
#include <stdint.h>

#include "fmha_decode_pieces.hpp"

extern "C" {

// out: shift, fine, parts, npv, total, full.
void pv_plan(int64_t batch, int units, int g, int max_rows, int d, int scattered, int forced_rows, int64_t* out) {
  const fmha_decode::PvPieces pv = fmha_decode::plan_pv_pieces(batch, units, g, max_rows, d, scattered != 0, forced_rows);
  const int64_t v[6] = {pv.shift, pv.fine, pv.parts, pv.npv, pv.total, pv.full};
  for (int i = 0; i < 6; ++i) out[i] = v[i];
}

// What the kernels make of the lengths: the size taken (as they add the rows
// up: in 32 bits, up to kOrderBatches batches), and the pieces of all batches
// and of the batch that has the most.
void pv_take(int64_t batch, int units, int g, int max_rows, int d, int scattered, int forced_rows, int uniform,
             const int32_t* lens, int64_t* shift, int64_t* all, int64_t* most) {
  const fmha_decode::PvPieces pv = fmha_decode::plan_pv_pieces(batch, units, g, max_rows, d, scattered != 0, forced_rows);
  int s = pv.shift;
  if (!uniform && batch <= fmha_decode::kOrderBatches) {
    int rows = 0;
    for (int64_t b = 0; b < batch; ++b) rows += fmha_decode::pv_counted_rows(lens[b], max_rows);
    s = fmha_decode::pv_device_shift(pv, rows);
  }
  *shift = s;
  *all = *most = 0;
  for (int64_t b = 0; b < batch; ++b) {
    // One length, or too many batches to add up: as many as the longest row has.
    const bool same = uniform || batch > fmha_decode::kOrderBatches;
    const int64_t n = fmha_decode::pv_row_pieces(same ? max_rows : lens[b], max_rows, s);
    *all += n;
    if (n > *most) *most = n;
  }
}

}  // extern "C"
