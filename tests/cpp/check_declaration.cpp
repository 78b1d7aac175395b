// Checks that a batch whose hierarchy could not be declared for want of memory
// runs as one without a hierarchy: the C API is built on stand-ins of the HIP
// runtime and of the kernels' launch functions (host memory, nothing runs), and
// each device allocation of spark_set_amr_grid fails in turn, in a first
// declaration and in one over an earlier hierarchy; so does each allocation of
// spark_batch_create before it.  Every pointer that a launch is handed has to be
// an allocation that is still there, and no launch returns the error of a call
// before it.  Prints "ok <cases>" or the first mismatch.
#include "../../flash-x_amd/csrc/spark_capi.cpp"

#include <cstdlib>

namespace {

std::map<void*, size_t> live;
int fail_at = -1;  // the allocation that fails (counted down), < 0: none
int allocations = 0;
int fills = 0, table_reads = 0, stages = 0;
bool bad = false;
hipError_t kept = hipSuccess;  // what hipGetLastError returns once, as after a launch

void expect(bool ok, const char* what) {
  if (!ok && !bad) std::printf("%s\n", what);
  bad = bad || !ok;
}

bool allocated(const void* p) {
  auto it = live.upper_bound(const_cast<void*>(p));
  if (it == live.begin()) return false;
  --it;
  return (const char*)p < (const char*)it->first + std::max<size_t>(1, it->second);
}

void check(const spark::PlainLaunch& L) {
  expect(allocated(L.meta) && (!L.blist || allocated(L.blist)) && allocated(L.flat), "a launch without its tables");
  expect(!L.blo || allocated(L.blo), "stage boxes that are not there");
  expect(!L.nbr || allocated(L.nbr), "a neighbour table that is not there");
  table_reads += L.nbr != nullptr || L.blo != nullptr;
}

}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  allocations++;
  *p = nullptr;
  if (fail_at >= 0 && fail_at-- == 0) return kept = hipErrorOutOfMemory;
  *p = std::calloc(1, std::max<size_t>(1, n));
  live[*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  expect(live.erase(p) == 1, "memory given back twice");
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemset(void* d, int v, size_t n) { std::memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return hipSuccess; }
hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = *t = size_t(64) << 30; return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 160 << 10;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)1; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = kept;
  kept = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t) { return "an error"; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
// not called
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorUnknown; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorUnknown; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipErrorUnknown; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipErrorUnknown; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) { return hipErrorUnknown; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorUnknown; }
}

namespace spark {
hipError_t plain_stage(const PlainLaunch& L, int, double, double, double, int) {
  check(L);
  expect(allocated(L.Sin) && allocated(L.Sout) && allocated(L.div.p), "a stage without its states");
  stages++;
  return hipGetLastError();
}
hipError_t plain_shock_detect(const PlainLaunch& L, double*, double*, int, const int64_t* nbr) {
  check(L);
  expect(!nbr || allocated(nbr), "a neighbour table that is not there");
  table_reads += nbr != nullptr;
  return hipSuccess;
}
hipError_t plain_set_scalar(hipStream_t, double* p, double) {
  expect(allocated(p), "no dt");
  return hipGetLastError();
}
hipError_t plain_correct(const PlainLaunch& L, double*, const unsigned char* f) {
  check(L);
  expect(!f || allocated(f), "face masks that are not there");
  return hipSuccess;
}
size_t plain_dt_part_size() { return 64; }
hipError_t amr_fill(const PlainLaunch& L, const AmrGrid& G, double*, const VarList&, int, const uint32_t* m, int) {
  check(L);
  expect(allocated(G.map) && allocated(G.org) && (!m || allocated(m)), "a hierarchy that is not there");
  fills++;
  return hipSuccess;
}
hipError_t amr_halo_copy(const PlainLaunch& L, const AmrGrid&, double*, const VarList&, int, const uint32_t* m) {
  check(L);
  expect(allocated(m), "sector masks that are not there");
  return hipSuccess;
}
hipError_t amr_flux_exchange(const PlainLaunch& L, const AmrGrid& G, double* const*, double* const*) {
  check(L);
  expect(allocated(G.map) && allocated(G.org), "a hierarchy that is not there");
  return hipSuccess;
}
size_t fused_lds_bytes(int, int tx, int ty) { return 64 * (size_t)(tx + 6) * (ty + 6); }
size_t fused_static_lds(int) { return 512; }
hipError_t fused_occupancy(int, size_t, int* n) { *n = 2; return hipSuccess; }
hipError_t fused_reset(hipStream_t, int* c) { expect(allocated(c), "no queue heads"); return hipSuccess; }
hipError_t fused_stage(const FusedArgs& A, int, size_t, hipStream_t) {
  expect(allocated(A.Sin) && allocated(A.Sout) && (!A.nbr || allocated(A.nbr)), "a fused stage without its tables");
  table_reads += A.nbr != nullptr;
  stages++;
  return hipGetLastError();
}
hipError_t noalloc_scratch_address(void** p) { *p = (void*)256; return hipSuccess; }
void xfer_release() {}
// not called
hipError_t plain_dt_part(const PlainLaunch&, const double*, void*, int) { return hipErrorUnknown; }
hipError_t plain_dt_final(hipStream_t, const DevParams&, const void*, int, int, double*, long long*, double*, int*, DtCtl*) {
  return hipErrorUnknown;
}
hipError_t plain_ug_fill(const PlainLaunch&, int, int, int, double*, const VarList&, int) { return hipErrorUnknown; }
hipError_t plain_set_int(hipStream_t, int*, int) { return hipErrorUnknown; }
hipError_t plain_aos_to_soa(hipStream_t, const BlockMeta*, int, int, const double*, const int64_t*, int, const int*, int,
                            double*) {
  return hipErrorUnknown;
}
hipError_t xfer_pack(const XferJob&, const double* const*, int, hipStream_t) { return hipErrorUnknown; }
hipError_t xfer_unpack(const XferJob&, double* const*, int, hipStream_t) { return hipErrorUnknown; }
}  // namespace spark

// 2 x 1 x 2 blocks, one of them refined: full and partial same-level halos
static spark_batch* make(int form, std::vector<int>& origins) {
  const int n = 10;
  spark_params p;
  spark_params_default(&p);
  p.ndim = 3;
  p.nguard = 10;
  p.nscalars = 1;
  p.flux_correct = 1;
  p.form = form;
  p.guard_mode = SPARK_GUARD_TELESCOPE;
  p.nunk_vars = SPARK_NPROP + 1;
  for (int v = 0; v < p.nunk_vars; v++) p.var_index[v] = v;
  std::vector<spark_block_desc> bl;
  origins.clear();
  auto add = [&](int level, int x, int y, int z) {
    bl.push_back(spark_block_desc{n, n, n, level, 1. / level, 1. / level, 1. / level});
    for (int o : {x, y, z}) origins.push_back(o * n);
  };
  for (int q = 0; q < 4; q++) {
    if (q == 3)
      for (int c = 0; c < 8; c++) add(2, 2 + c % 2, c / 2 % 2, 2 + c / 4);
    else
      add(1, q % 2, 0, q / 2);
  }
  spark_batch* b = nullptr;
  if (spark_batch_create(&p, (int)bl.size(), bl.data(), &b) != SPARK_OK) return nullptr;
  spark_set_option(b, SPARK_OPT_AUTOTUNE, 0);
  return b;
}

int main() {
  const int bc[3] = {SPARK_BC_PERIODIC, SPARK_BC_OUTFLOW, SPARK_BC_REFLECT};
  int cases = 0;
  if (spark_init(0) != SPARK_OK) return std::printf("spark_init\n"), 1;
  std::vector<int> org;
  for (int form : {SPARK_FORM_PLAIN_FP64, SPARK_FORM_BATCHED_FP64, SPARK_FORM_FP32_FLUX})
    for (int k = 0;; k++, cases++) {
      // the pool of the divergence terms is left out where it cannot be had
      const size_t before = live.size();
      fail_at = k;
      spark_batch* b = make(form, org);
      const bool failed = fail_at < 0;
      fail_at = -1;
      expect(kept == hipSuccess, "an error that is kept");
      if (!b) {
        expect(failed && live.size() == before, "a batch that failed holds memory");
        continue;
      }
      expect(spark_hydro_step(b, 1e-3, 1e-3) == SPARK_OK, "a step that fails");
      spark_batch_destroy(b);
      if (bad) return std::printf("form %d, allocation %d of a batch\n", form, k), 1;
      if (!failed) break;
    }
  for (int form : {SPARK_FORM_PLAIN_FP64, SPARK_FORM_BATCHED_FP64, SPARK_FORM_FP32_FLUX})
    for (bool over : {false, true}) {
      auto declare = [&](spark_batch* b) { return spark_set_amr_grid(b, 2, 1, 2, org.data(), bc); };
      auto step = [&](spark_batch* b) {
        fills = table_reads = stages = 0;
        const int rc = spark_hydro_step(b, 1e-3, 1e-3);
        expect(rc == SPARK_OK && stages > 0, "a step that fails");
      };
      for (int k = 0;; k++) {
        spark_batch* b = make(form, org);
        if (!b) return std::printf("no batch\n"), 1;
        if (over) {
          expect(declare(b) == SPARK_OK, "the first declaration");
          step(b);
        }
        fail_at = k;
        allocations = 0;
        const int rc = declare(b);
        fail_at = -1;
        if (rc == SPARK_OK) {
          expect(allocations == k, "a failed allocation without an error");
          step(b);
          expect(fills > 0 && table_reads > 0, "a hierarchy that is not used");
          spark_batch_destroy(b);
          break;
        }
        expect(spark_fill_guardcells(b) == SPARK_ERR_STATE, "a guard fill without a hierarchy");
        step(b);
        expect(fills == 0 && table_reads == 0, "tables of a hierarchy that was not declared");
        expect(declare(b) == SPARK_OK, "a declaration after one that failed");
        step(b);
        expect(fills > 0 && table_reads > 0, "a hierarchy that is not used");
        spark_batch_destroy(b);
        if (bad) return std::printf("form %d, allocation %d, over %d\n", form, k, (int)over), 1;
        cases++;
      }
    }
  expect(live.empty(), "memory not given back");
  if (bad) return 1;
  std::printf("ok %d\n", cases);
  return 0;
}
