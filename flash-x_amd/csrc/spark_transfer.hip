// spark_transfer.hip -- the staged, pipelined transfers of spark_transfer.hpp.
//
// Bound by PCIe (57 GB/s each way from pinned memory).  Pageable copies of
// one block at a time reached 28 GB/s to the device and 17.5 GB/s back, and
// an interior-only unpack uploaded and downloaded every guard-celled block;
// here it moves the interior cells once.  576 blocks of 16^3, 10 guard cells
// and 19 variables: interior unpack 390 -> 9.4 ms; 160 mixed blocks (0.73 GB):
// pack 29 -> 13 ms, interior unpack 72 -> 2.9 ms.
#include <string.h>

#include <algorithm>
#include <atomic>
#include <deque>
#include <exception>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

#include "spark_transfer.hpp"
#include "spark_workers.hpp"

namespace spark {
namespace {

__device__ __forceinline__ int64_t seg_cell(const BlockMeta& m, int ng, int ndim, int interior, int64_t t) {
  if (!interior) return box_cell(m, t);
  const int i = (int)(t % m.nx);
  const int64_t row = t / m.nx;
  const int j = (int)(row % m.ny), k = (int)(row / m.ny);
  return (ng + i) + (int64_t)m.PX * (j + (ndim > 1 ? ng : 0) + (int64_t)m.NY * (k + (ndim > 2 ? ng : 0)));
}

// One thread per cell: the state side is coalesced; a wave's tuples are one
// contiguous stretch of staging memory whose lines its loop over the
// variables uses up from cache.
__global__ void __launch_bounds__(256) k_unstage(const XferSeg* __restrict__ segs, const BlockMeta* __restrict__ meta,
                                                 const double* __restrict__ stage, int width,
                                                 const int* __restrict__ slot, int nvar, double* __restrict__ pool) {
  const XferSeg s = segs[blockIdx.y];
  const BlockMeta m = meta[s.blk];
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < s.ncell; t += (int64_t)gridDim.x * blockDim.x) {
    const double* src = stage + (s.at + t) * width;
    double* dst = pool + m.base + box_cell(m, s.cell0 + t);
    for (int v = 0; v < nvar; v++) dst[v * m.cstride] = src[slot[v]];
  }
}

__global__ void __launch_bounds__(256) k_stage(const XferSeg* __restrict__ segs, const BlockMeta* __restrict__ meta,
                                               const double* __restrict__ pool, int ng, int ndim, int interior,
                                               int width, const int* __restrict__ slot, int nvar,
                                               double* __restrict__ stage) {
  const XferSeg s = segs[blockIdx.y];
  const BlockMeta m = meta[s.blk];
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < s.ncell; t += (int64_t)gridDim.x * blockDim.x) {
    const double* src = pool + m.base + seg_cell(m, ng, ndim, interior, s.cell0 + t);
    double* dst = stage + (s.at + t) * width;
    for (int v = 0; v < nvar; v++) dst[slot[v]] = src[v * m.cstride];
  }
}

constexpr size_t SLOT_BYTES = size_t(8) << 20;
constexpr int SLOT_SEGS = 1024;  // segments of a chunk

struct Slot {
  unsigned char* host = nullptr;
  unsigned char* dev = nullptr;
  hipStream_t stream = nullptr;
  hipEvent_t done = nullptr;
  bool used = false;
};

struct Staging {
  std::mutex mu;
  int device = -1;
  size_t bytes = 0;
  Slot slot[XFER_SLOTS];
  hipEvent_t before = nullptr;

  void release() {
    for (Slot& s : slot) {
      if (s.stream) {
        (void)hipStreamSynchronize(s.stream);
        (void)hipStreamDestroy(s.stream);
      }
      if (s.done) (void)hipEventDestroy(s.done);
      if (s.host) (void)hipHostFree(s.host);
      if (s.dev) (void)hipFree(s.dev);
      s = Slot();
    }
    if (before) (void)hipEventDestroy(before);
    before = nullptr;
    device = -1;
    bytes = 0;
  }
  hipError_t ensure(int dev, size_t need) {
    if (device == dev && bytes >= need) return hipSuccess;
    release();
    hipError_t e = hipEventCreateWithFlags(&before, hipEventDisableTiming);
    for (Slot& s : slot) {
      if (e == hipSuccess) e = hipHostMalloc((void**)&s.host, need, hipHostMallocDefault);
      if (e == hipSuccess) e = hipMalloc((void**)&s.dev, need);
      if (e == hipSuccess) e = hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking);
      if (e == hipSuccess) e = hipEventCreateWithFlags(&s.done, hipEventDisableTiming);
    }
    if (e != hipSuccess) {
      release();
      return e;
    }
    device = dev;
    bytes = need;
    return hipSuccess;
  }
};
Staging g_staging;

// A slot's area: the variable map, the segments, then (256-byte aligned) the
// tuples.  The map and the segments travel with the tuples of a pack.
struct Area {
  size_t seg_at, data_at;
  Area(int nvar) {
    seg_at = (sizeof(int) * (size_t)nvar + 255) / 256 * 256;
    data_at = (seg_at + sizeof(XferSeg) * SLOT_SEGS + 255) / 256 * 256;
  }
};

struct Chunk {
  size_t seg0;
  int nseg;
  int64_t cells, longest;
};

struct Plan {
  std::vector<XferSeg> segs;
  std::vector<Chunk> chunks;
};

Plan make_plan(const XferJob& j, int64_t cells_per_chunk) {
  Plan p;
  Chunk c{0, 0, 0, 0};
  auto close = [&]() {
    if (c.nseg) p.chunks.push_back(c);
    c = Chunk{p.segs.size(), 0, 0, 0};
  };
  for (int b = 0; b < j.nblk; b++) {
    const BlockMeta& m = j.meta_h[b];
    const int64_t total = j.interior ? (int64_t)m.nx * m.ny * m.nz : (int64_t)m.NX * m.NY * m.NZ;
    for (int64_t done = 0; done < total;) {
      if (c.cells == cells_per_chunk || c.nseg == SLOT_SEGS) close();
      const int64_t n = std::min(total - done, cells_per_chunk - c.cells);
      p.segs.push_back(XferSeg{done, n, c.cells, b, 0});
      c.nseg++;
      c.cells += n;
      c.longest = std::max(c.longest, n);
      done += n;
    }
  }
  close();
  return p;
}

// the cells of a segment between the host block and packed tuples
void copy_in(const XferJob& j, const double* block, const XferSeg& s, double* tuples) {
  memcpy(tuples + s.at * j.nunk, block + s.cell0 * j.nunk, sizeof(double) * (size_t)s.ncell * j.nunk);
}
void copy_out(const XferJob& j, double* block, const XferSeg& s, const double* tuples, bool whole) {
  const BlockMeta& m = j.meta_h[s.blk];
  const int width = whole ? j.nunk : j.nvar;
  const int64_t row = j.interior ? m.nx : s.cell0 + s.ncell;  // runs of consecutive host cells
  for (int64_t t = s.cell0; t < s.cell0 + s.ncell;) {
    const int64_t n = std::min(row - t % row, s.cell0 + s.ncell - t);
    int64_t c = t;
    if (j.interior) {
      const int64_t r = t / m.nx;
      c = j.ng + t % m.nx + (int64_t)m.NX * (r % m.ny + (j.ndim > 1 ? j.ng : 0) +
                                            (int64_t)m.NY * (r / m.ny + (j.ndim > 2 ? j.ng : 0)));
    }
    const double* src = tuples + (s.at + t - s.cell0) * width;
    double* dst = block + c * j.nunk;
    if (whole) {
      memcpy(dst, src, sizeof(double) * (size_t)n * width);
    } else {
      for (int64_t q = 0; q < n; q++)
        for (int v = 0; v < j.nvar; v++) dst[q * j.nunk + j.var_index[v]] = src[q * j.nvar + v];
    }
    t += n;
  }
}

unsigned grid_x(int64_t cells) { return (unsigned)std::min<int64_t>(512, (cells + 255) / 256); }

hipError_t transfer(const XferJob& j, double* const* host, bool pack, int device, hipStream_t stream) {
  std::lock_guard<std::mutex> lock(g_staging.mu);
  // Every unk slot is a variable of the state, each once: whole tuples move.
  // Otherwise an unpack moves the variables only and the host copy leaves
  // the other slots alone; a pack always moves the host's whole tuples.
  std::vector<char> seen(j.nunk, 0);
  bool whole = j.nvar == j.nunk;
  for (int v = 0; v < j.nvar; v++) {
    if (seen[j.var_index[v]]) whole = false;
    seen[j.var_index[v]] = 1;
  }
  const int width = pack || whole ? j.nunk : j.nvar;
  const Area area(j.nvar);
  const size_t tuple = sizeof(double) * (size_t)width;
  hipError_t e = hipSetDevice(device);
  if (e == hipSuccess) e = g_staging.ensure(device, std::max(SLOT_BYTES, area.data_at + tuple));
  if (e != hipSuccess) return e;
  int64_t cells = 0;
  for (int b = 0; b < j.nblk; b++) {
    const BlockMeta& m = j.meta_h[b];
    cells += j.interior ? (int64_t)m.nx * m.ny * m.nz : (int64_t)m.NX * m.NY * m.NZ;
  }
  // From 4 MiB on, four threads (one copies 30 GB/s, half of what PCIe
  // takes); below, starting them costs more than they save and the calling
  // thread keeps all slots in flight.  About eight chunks, so that the ends of
  // the pipeline are short, of at least 256 KiB, where DMA reaches half speed.
  const double bytes = (double)cells * tuple;
  const int hw = std::max(1u, std::thread::hardware_concurrency());
  const int workers = bytes >= 4 << 20 ? std::min(XFER_SLOTS, hw) : 1;
  const int64_t most = (int64_t)((g_staging.bytes - area.data_at) / tuple);
  const int64_t even = (cells + 7) / 8, least = (int64_t)((size_t(256) << 10) / tuple) + 1;
  const Plan plan = make_plan(j, std::max<int64_t>(1, std::min(most, std::max(even, least))));
  std::vector<int> slots(j.nvar);
  for (int v = 0; v < j.nvar; v++) slots[v] = width == j.nunk ? j.var_index[v] : v;

  e = hipEventRecord(g_staging.before, stream);
  for (Slot& s : g_staging.slot)
    if (e == hipSuccess) e = hipStreamWaitEvent(s.stream, g_staging.before, 0);
  if (e != hipSuccess) return e;

  std::atomic<size_t> next{0};
  std::atomic<int> failed{(int)hipSuccess};
  auto fail = [&](hipError_t err) {
    int ok = (int)hipSuccess;
    failed.compare_exchange_strong(ok, (int)err);
  };
  // starts chunk c on a slot: header and (pack) tuples to the device, the
  // transpose, (unpack) the tuples back
  auto start = [&](Slot& s, const Chunk& c) -> hipError_t {
    hipError_t r = s.used ? hipEventSynchronize(s.done) : hipSuccess;
    if (r != hipSuccess) return r;
    s.used = true;
    const XferSeg* segs = plan.segs.data() + c.seg0;
    memcpy(s.host, slots.data(), sizeof(int) * slots.size());
    memcpy(s.host + area.seg_at, segs, sizeof(XferSeg) * c.nseg);
    const size_t data = tuple * (size_t)c.cells;
    if (pack)
      for (int q = 0; q < c.nseg; q++)
        copy_in(j, host[segs[q].blk], segs[q], reinterpret_cast<double*>(s.host + area.data_at));
    const size_t up = pack ? area.data_at + data : area.seg_at + sizeof(XferSeg) * c.nseg;
    if ((r = hipMemcpyAsync(s.dev, s.host, up, hipMemcpyHostToDevice, s.stream)) != hipSuccess) return r;
    const XferSeg* segs_d = reinterpret_cast<const XferSeg*>(s.dev + area.seg_at);
    double* tuples_d = reinterpret_cast<double*>(s.dev + area.data_at);
    const int* slots_d = reinterpret_cast<const int*>(s.dev);
    const dim3 grid(grid_x(c.longest), c.nseg);
    if (pack)
      hipLaunchKernelGGL(k_unstage, grid, dim3(256), 0, s.stream, segs_d, j.meta_d, tuples_d, width, slots_d, j.nvar,
                         j.pool);
    else
      hipLaunchKernelGGL(k_stage, grid, dim3(256), 0, s.stream, segs_d, j.meta_d, j.pool, j.ng, j.ndim, j.interior,
                         width, slots_d, j.nvar, tuples_d);
    if ((r = hipGetLastError()) != hipSuccess) return r;
    if (!pack && (r = hipMemcpyAsync(s.host + area.data_at, tuples_d, data, hipMemcpyDeviceToHost, s.stream)) != hipSuccess)
      return r;
    return hipEventRecord(s.done, s.stream);
  };
  auto work = [&](int w) {
    hipError_t r = hipSetDevice(device);
    std::deque<std::pair<Slot*, const Chunk*>> flying;  // unpack: chunks on their way, oldest first
    int turn = 0;
    const int mine = (XFER_SLOTS - w + workers - 1) / workers;
    while (r == hipSuccess && failed.load() == (int)hipSuccess) {
      if (pack || (int)flying.size() < mine) {
        const size_t c = next.fetch_add(1);
        if (c < plan.chunks.size()) {
          Slot& s = g_staging.slot[w + workers * (turn++ % mine)];
          r = start(s, plan.chunks[c]);
          if (!pack && r == hipSuccess) flying.push_back({&s, &plan.chunks[c]});
          continue;
        }
        if (flying.empty()) break;
      }
      const auto f = flying.front();
      flying.pop_front();
      if ((r = hipEventSynchronize(f.first->done)) != hipSuccess) break;
      for (int q = 0; q < f.second->nseg; q++) {
        const XferSeg& s = plan.segs[f.second->seg0 + q];
        copy_out(j, host[s.blk], s, reinterpret_cast<const double*>(f.first->host + area.data_at), whole);
      }
    }
    if (r != hipSuccess) fail(r);
  };
  run_workers(workers, [&](int w) {
    try {
      work(w);
    } catch (const std::exception&) {
      fail(hipErrorOutOfMemory);
    }
  });
  e = (hipError_t)failed.load();
  for (Slot& s : g_staging.slot) {
    if (!s.used) continue;
    if (e == hipSuccess) e = hipStreamWaitEvent(stream, s.done, 0);
    else (void)hipStreamSynchronize(s.stream);
  }
  return e;
}

}  // namespace

hipError_t xfer_pack(const XferJob& j, const double* const* host, int device, hipStream_t stream) {
  return transfer(j, const_cast<double* const*>(host), true, device, stream);
}

hipError_t xfer_unpack(const XferJob& j, double* const* host, int device, hipStream_t stream) {
  return transfer(j, host, false, device, stream);
}

void xfer_release() {
  std::lock_guard<std::mutex> lock(g_staging.mu);
  g_staging.release();
}

}  // namespace spark
