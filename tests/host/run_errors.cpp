// A run that fails after its first launch leaves nothing in flight: the next run
// writes its queues to the host memory that the failed one's first kernel reads,
// and a larger plan frees it.  xt_host.cpp runs here over a stand-in for the HIP
// runtime that counts what is queued on the stream and fails the call it is told
// to.  Built and run by tests/test_run_errors.py.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../exachem_amd/csrc/xt_device.h"
#include "../../include/exachem_t.h"

namespace {
enum Fault { kNone, kSpatial, kReduce, kFirstEvent, kSecondEvent, kGraphLaunch, kQuery };
Fault fault = kNone;
int   pending = 0, events = 0, freed_in_flight = 0;
bool  capturing = false;

hipError_t queued() {
  if(!capturing) pending++;
  return hipSuccess;
}
int launched(bool failing) { return failing ? (int) hipErrorLaunchFailure : (int) queued(); }
hipError_t freed(void* p) {
  freed_in_flight += pending != 0;
  std::free(p);
  return hipSuccess;
}
template<class T>
T handle() {
  return reinterpret_cast<T>(std::malloc(1));
}
}  // namespace

extern "C" {
hipError_t  hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t  hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t  hipSetDevice(int) { return hipSuccess; }
hipError_t  hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 100000, hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "injected"; }
hipError_t  hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  std::memset(p, 0, sizeof *p);
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 4;
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* a, size_t* b) { return *a = *b = 1ull << 40, hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { return *p = std::calloc(n ? n : 1, 1), hipSuccess; }
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }  // waits for the device
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { return freed(p); }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return *e = handle<hipEvent_t>(), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return std::free(e), hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0.f, hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) {
  events++;
  return (fault == kFirstEvent && events == 1) || (fault == kSecondEvent && events == 2) ? hipErrorUnknown
                                                                                          : hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = handle<hipStream_t>(), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return std::free(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return pending = 0, hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) {
  return fault == kQuery ? hipErrorUnknown : (pending = 0, hipSuccess);
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return capturing = true, hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  capturing = false;
  return *g = handle<hipGraph_t>(), hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { return std::free(g), hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t g) { return std::free(g), hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  return *e = handle<hipGraphExec_t>(), hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
  return fault == kGraphLaunch ? hipErrorUnknown : queued();
}
int xt_mlp_predict(xt_mlp*, long, const float*, float*) { std::abort(); }
int xt_mlp_train(xt_mlp*, long, const float*, const float*, int, float, float*) { std::abort(); }
}

namespace xt {
int build_split(const SpatialBufs&, int, int, const int*, int, const int*, int, SplitBufs&, void*) { return 0; }
int build_part_scales(const TaskDev*, int, const MixedDev&, float*, void*) { return 0; }
int build_operands(int, int, double*, double*, double*&, SpatialBufs&, void*) { return 0; }
int build_xva(int, int, SpatialBufs&, void*) { return 0; }
int cholesky_integrals(int, int, long, const double*, double*, double*, double*, void*) { std::abort(); }
int launch_vvoo_asym(const double*, int, int, double*, int* groups, void*) { return *groups = 0; }
int launch_begin(unsigned long long*, long, unsigned long long*, const unsigned long long*, long, long, long, void*) {
  return launched(false);
}
int launch_spatial_fp64(const SpatialDev&, const RunDev&, int, void*) { return launched(fault == kSpatial); }
int launch_spatial_mixed(const MixedDev&, const RunDev&, int, void*) { return launched(fault == kSpatial); }
int launch_reduce(const TaskDev*, int, const int*, const int*, const unsigned long long*, const unsigned long long*,
                  double*, double*, double*, void*) {
  return launched(fault == kReduce);
}
int launch_packed_fp64(const PackedArgs&, void*) { std::abort(); }
int launch_packed_fp64_noalloc(PackedArgs&, const int*, int, void*, void*) { std::abort(); }
int launch_gather(const GatherDesc*, int, long, const GatherSrc&, const GatherDst&, void*) { std::abort(); }
int launch_expand_t(const GatherSrc&, double*, double*, void*) { std::abort(); }
}  // namespace xt

int main() {
  const int small[1] = {2}, vir[1] = {3}, occ2[2] = {1, 1}, vir2[3] = {1, 1, 1};
  for(int graph = 0; graph < 2; graph++)
    for(int prec = 0; prec < 2; prec++)
      for(int f = kSpatial; f <= kQuery; f++) {
        xt_ctx* c = nullptr;
        double  e[2];
        if(xt_create(0, &c) || xt_set_tiling(c, 2, 3, 1, small, 1, vir, 0) || xt_synth_upload(c, 1, 0.05, 1e-3))
          return std::printf("run_errors: setup: %s\n", xt_last_error()), 1;
        xt_opts o;
        xt_default_opts(&o);
        o.precision   = prec;
        o.use_graph   = graph;
        o.progress_ms = f == kQuery ? 1000 : 0;
        if(xt_prepare(c, prec)) return std::printf("run_errors: prepare: %s\n", xt_last_error()), 1;
        fault  = (Fault) f;
        events = 0;
        const int rc = xt_run(c, &o, e, nullptr, nullptr);
        fault = kNone;
        if(rc == XT_OK && !(f == kGraphLaunch && !graph))
          return std::printf("run_errors: fault %d (graph %d) was not reported\n", f, graph), 1;
        if(pending) return std::printf("run_errors: %d operations in flight after fault %d (graph %d)\n", pending, f, graph), 1;
        if(xt_run(c, &o, e, nullptr, nullptr)) return std::printf("run_errors: next run: %s\n", xt_last_error()), 1;
        if(xt_set_tiling(c, 2, 3, 2, occ2, 3, vir2, 0) || xt_run(c, &o, e, nullptr, nullptr) || xt_destroy(c))
          return std::printf("run_errors: larger plan: %s\n", xt_last_error()), 1;
        if(freed_in_flight) return std::printf("run_errors: host memory freed in flight\n"), 1;
      }
  std::printf("run_errors: ok\n");
  return 0;
}
