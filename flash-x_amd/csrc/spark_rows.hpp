// spark_rows.hpp -- row layout of the state pools (host code).
#pragma once
#include <stdint.h>

#include <initializer_list>

namespace spark {

// Rows of a block's guard-celled box in the pools: `pitch` doubles apart, the
// box `lead` doubles into its place, so that every row's first interior cell
// starts a 128-byte line (a 64-byte half line where full lines would cost more
// than a third of the memory; rows stay packed where that does too).  16 cells
// of a packed 36-cell row lie across two lines or three halves and share them
// with guard cells, and the lines moved bound the sweeps of packed rows.
// 576 leaves of 16^3 with 8 scalars, FP64: the sweeps over the interiors
// fetched 2.6 and wrote 1.3 GB per stage packed, 1.4 and 1.0 GB aligned.
struct RowPad { int pitch, lead; };
inline RowPad row_pad(int NX, int ng) {
  for (int a : {16, 8}) {
    const int pitch = (NX + a - 1) / a * a;
    if (3 * pitch <= 4 * NX) return RowPad{pitch, (a - ng % a) % a};
  }
  return RowPad{NX, 0};
}

// Whether a batch pads its rows: where the padded state takes no more than 3/8
// of the memory that is free.  Padding then never keeps a batch from fitting,
// and what it takes from the batches after it is at most 3/32 of that memory.
// The bound is not higher because memory given back has to be cleared before it
// is allocated again: the batch after one of the same size (a regrid) takes
// 24 ms to create while both fit into the GPU's 288 GB at once, 1.3 s and more
// beyond (4384 leaves of 16^3 with 8 scalars, 107 GB packed and 138 GB padded).
// cells: of all blocks' padded boxes; fields: doubles per cell.
inline bool pad_rows(int64_t cells, int64_t fields, int64_t free_bytes) {
  return cells * fields * (int64_t)sizeof(double) <= free_bytes / 8 * 3;
}

// Whether the FP64 sweeps get a pool of their own for their divergence terms:
// where it takes no more than a quarter of the memory its batch leaves.  Without
// it they keep the terms in the stage buffers, which is as fast for most
// batches; on 4384 leaves of 16^3 with 8 scalars the x sweep, then writing the
// buffer beside the one it reads, takes 13.8 instead of 11.3 ms a step.
inline bool div_pool(int64_t doubles, int64_t free_bytes) {
  return doubles * (int64_t)sizeof(double) <= free_bytes / 4;
}

}  // namespace spark
