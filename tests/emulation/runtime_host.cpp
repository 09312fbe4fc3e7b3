// lk::Runtime's host code on a HIP runtime of host memory that counts its
// allocations and fails them on request; launches check that what they are
// given is allocated and compute nothing.
#include <cstdio>
#include <cstdlib>

#include "../../libkriging_amd/csrc/lk_runtime.cpp"

#include "../../libkriging_amd/csrc/model_io.cpp"

namespace {
std::map<char*, size_t> live;
int errors = 0, countdown = -1;  // allocations that still succeed (-1: all)
hipError_t last = hipSuccess;    // until it is asked for
intptr_t handles = 0;            // streams and graphs made
bool capturing = false;
int captures = 0, events_captured = 0;
std::vector<hipStream_t> launched;  // streams of the graph launches

hipError_t take(void** p, size_t bytes) {
  if (countdown == 0) return last = hipErrorOutOfMemory;
  if (countdown > 0) --countdown;
  *p = std::calloc(1, bytes ? bytes : 1);
  live[(char*)*p] = bytes;
  return hipSuccess;
}
hipError_t give(void* p) {
  if (p == nullptr) return hipSuccess;
  if (live.erase((char*)p) == 0) {
    ++errors;  // not allocated, or freed before
    return hipErrorInvalidValue;
  }
  return hipSuccess;  // (kept, so that a use of it can be counted)
}
void expect(const void* p, size_t bytes) {
  auto it = live.upper_bound((char*)p);
  if (it == live.begin() || (char*)p + bytes > (--it)->first + it->second) ++errors;
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return take(p, n); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return take(p, n); }
hipError_t hipFree(void* p) { return give(p); }
hipError_t hipHostFree(void* p) { return give(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemcpy2D(void*, size_t, const void*, size_t, size_t, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemcpy2DAsync(void*, size_t, const void*, size_t, size_t, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = (hipEvent_t)1, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* f, hipEvent_t, hipEvent_t) { return *f = 0, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return events_captured += capturing, hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = (hipStream_t)++handles, hipSuccess; }
hipError_t hipExtStreamCreateWithCUMask(hipStream_t* s, uint32_t, const uint32_t*) { return *s = (hipStream_t)++handles, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return events_captured += capturing, hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return ++captures, capturing = true, hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return capturing = false, *g = (hipGraph_t)1, hipSuccess; }
hipError_t hipGraphCreate(hipGraph_t* g, unsigned) { return *g = (hipGraph_t)1, hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) { return *e = (hipGraphExec_t)1, hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) { return launched.push_back(s), hipSuccess; }
hipError_t hipGraphAddChildGraphNode(hipGraphNode_t*, hipGraph_t, const hipGraphNode_t*, size_t, hipGraph_t) { return hipSuccess; }
hipError_t hipGraphAddEventRecordNode(hipGraphNode_t*, hipGraph_t, const hipGraphNode_t*, size_t, hipEvent_t) { return hipSuccess; }
}

namespace lk {
hipError_t noalloc_scratch(int, char** p) { return *p = nullptr, hipSuccess; }
int trtri_levels(int) { return 0; }
// every launch of a batch: its tables and its slots' memory are allocated
static hipError_t check(const Batch& b) {
  expect(b.slots, sizeof(Slot) * b.nslots);
  expect(b.params, sizeof(SlotParams) * b.nslots);
  expect(b.out, sizeof(SlotOut) * b.nslots);
  expect(b.host_params, sizeof(SlotParams) * b.nslots);
  expect(b.host_out, sizeof(SlotOut) * b.nslots);
  if (errors > 0) return hipGetLastError();
  for (int s = 0; s < b.nslots; ++s) {
    const Slot& S = b.slots[s];
    expect(S.X, sizeof(double) * S.n * S.d);
    expect(S.A, sizeof(double) * S.npad * S.npad);
    expect(S.W, sizeof(double) * S.npad * S.npad);
    expect(S.V, sizeof(double) * S.npad * v_cols(S.p));
    expect(S.red, sizeof(double) * red_size(S.nblk));
  }
  return hipGetLastError();
}
#define LAUNCH(name) hipError_t name(const Batch& b) { return check(b); }
LAUNCH(launch_build) LAUNCH(launch_gls) LAUNCH(launch_loo_g) LAUNCH(launch_loo_bs) LAUNCH(launch_loo_bw)
LAUNCH(launch_loo_wv) LAUNCH(launch_solve_e) LAUNCH(launch_solve_x) LAUNCH(launch_solve_fy)
LAUNCH(launch_loo_value) LAUNCH(launch_params_in) LAUNCH(launch_rinv_store) LAUNCH(launch_trtri_base)
LAUNCH(launch_finalize_ll) LAUNCH(launch_lmp_adjoint) LAUNCH(launch_loo_adjoint) LAUNCH(launch_results_out)
LAUNCH(launch_finalize_grad) LAUNCH(launch_lauum_adjoint) LAUNCH(launch_loo_finalize_grad)
hipError_t launch_potrf_chain(const Batch& b, int, int) { return check(b); }
hipError_t launch_potrf_rows(const Batch& b, int, int) { return check(b); }
hipError_t launch_trtri_level(const Batch& b, int, int) { return check(b); }
hipError_t launch_potrf_update(const Batch& b, int, int, int, int) { return check(b); }
hipError_t launch_potrf_update_trailing(const Batch& b, int, int, int) { return check(b); }
hipError_t launch_potrf_update_persistent(const Batch& b, int, int, int, int, int) { return check(b); }
hipError_t launch_schur(const SchurArgs&, hipStream_t) { return hipSuccess; }
hipError_t launch_block_assemble(const BlockAssembleArgs&, hipStream_t) { return hipSuccess; }
hipError_t launch_trmm_lower(const double*, const double*, double*, int, int, hipStream_t) { return hipSuccess; }
}  // namespace lk

// n-point designs of one dimension, evaluated in batches of one design
struct Bench {
  lk::Runtime rt{0};
  std::vector<double> x = std::vector<double>(300, 0.5), g = std::vector<double>(1, 0.3);
  int design(int n) { return rt.add_problem(x.data(), n, 1, x.data(), x.data(), 1, 0, 0); }
  void batch(int id, int items) {
    std::vector<lk::EvalRequest> r(items);
    for (auto& q : r) {
      q.problem = id;
      q.gamma = g.data();
      q.gamma_n = 1;
    }
    std::vector<lk::EvalResult> res;
    rt.evaluate(r, true, res);
  }
};

// A batch, then one that needs a larger pool and larger tables and whose
// allocation number `fail` (from 0) fails, then the first batch, another that
// fits the old pool, and the large one.  Returns the accesses to and frees of
// memory that is not allocated, + 1000 per block left at the end; -1 when no
// allocation failed.
static int failed_growth(int fail) {
  bool threw = false;
  {
    Bench t;
    t.rt.use_graph = false;
    const int a = t.design(100), b = t.design(60);
    auto batch = [&](int id, int items) { t.batch(id, items); };
    batch(a, 1);
    countdown = fail;
    try {
      batch(a, 9);
    } catch (const std::exception&) {
      threw = true;
    }
    countdown = -1;
    batch(a, 1);
    batch(b, 1);
    batch(a, 9);
    batch(a, 9);
  }
  return threw ? errors + 1000 * (int)live.size() : -1;
}

// Graphs of batches in parts: "captures events-in-captures launches
// distinct-streams" after a batch in four parts, after the same again, and
// after another design in two
static void split_batches() {
  Bench t;
  auto report = [&] {
    std::sort(launched.begin(), launched.end());
    const int streams = int(std::unique(launched.begin(), launched.end()) - launched.begin());
    std::printf("%d %d %d %d\n", captures, events_captured, (int)launched.size(), streams);
    launched.clear();
    captures = 0;
  };
  const int a = t.design(100), b = t.design(200);
  t.batch(a, 32);
  report();
  t.batch(a, 32);
  report();
  t.batch(b, 16);
  report();
}

int main(int, char** argv) {
  if (std::string(argv[1]) == "split")
    split_batches();
  else
    std::printf("%d\n", failed_growth(std::atoi(argv[1])));
  return 0;
}
