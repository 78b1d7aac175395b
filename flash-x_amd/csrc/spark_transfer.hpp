// spark_transfer.hpp -- host unk blocks <-> device state pools.
//
// A transfer is cut into chunks of at most one staging slot, a chunk into
// segments (consecutive cells of one block's box, or of its interior).  Each
// slot has pinned host memory, device memory and a stream of its own, so one
// chunk's host copy, another's DMA and a third's transpose run side by side.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "spark_launch.hpp"
#include "spark_physics.hpp"

namespace spark {

// cells [cell0, cell0 + ncell) of block blk's box (x fastest); their tuples
// start at tuple `at` of the chunk's staging area
struct XferSeg {
  int64_t cell0, ncell, at;
  int blk, pad;
};

struct XferJob {
  const BlockMeta* meta_h;  // host and device block tables
  const BlockMeta* meta_d;
  int nblk, ng, ndim, nvar, nunk;
  const int* var_index;     // host: unk slot of each variable
  double* pool;
  int interior;             // unpack: the interior cells only
};

// Staging of one device, shared by every batch and held between transfers:
// XFER_SLOTS x (pinned + device) areas.  Transfers take turns (the calls
// lock), the caller's stream is ordered before and after them.
constexpr int XFER_SLOTS = 4;

// host blocks -> pool; returns when the host blocks have been read (the
// device work is ordered before later work on `stream`)
hipError_t xfer_pack(const XferJob& j, const double* const* host, int device, hipStream_t stream);
// pool -> host blocks, after earlier work on `stream`; returns when done
hipError_t xfer_unpack(const XferJob& j, double* const* host, int device, hipStream_t stream);
// gives the staging back
void xfer_release();

}  // namespace spark
