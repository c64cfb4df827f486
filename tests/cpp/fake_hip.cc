// A host-only stand-in for the HIP runtime, loaded in front of the built
// library (same SONAME): "device" memory is zeroed host memory, copies are
// memcpy, kernels do not run.  Every launch is logged by its kernel's name; a
// launch can be made to fail, and a clock that the launches advance gives the
// events their times, so that the host code around the kernels runs without
// a GPU.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

namespace {
std::map<const void*, std::string> g_kernels;  // host stub -> device symbol
std::map<const void*, void*> g_vars;
std::string g_log;            // one line per launch, copy and wait
std::string g_fail;           // part of a kernel's name whose next launch fails
std::vector<std::pair<std::string, float>> g_cost;  // name part -> ms of a launch
double g_clock = 0.0;
hipError_t g_last = hipSuccess;
struct Event {
  double at = 0.0;
};
struct CallConfig {
  dim3 g, b;
  size_t sh;
  hipStream_t s;
} g_call;

hipError_t result(hipError_t e) {
  if (e != hipSuccess) g_last = e;
  return e;
}
}  // namespace

extern "C" {

// ---- control
void fake_hip_reset() {
  g_log.clear();
  g_fail.clear();
  g_cost.clear();
  g_last = hipSuccess;
}
const char* fake_hip_log() { return g_log.c_str(); }
void fake_hip_fail(const char* part) { g_fail = part; }
void fake_hip_cost(const char* part, float ms) { g_cost.push_back({part, ms}); }

// ---- registration and launches
void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* stub, char*, const char* name, unsigned, void*,
                           void*, void*, void*, int*) {
  g_kernels[stub] = name;
}
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t size, int, int) {
  g_vars[var] = std::calloc(1, size);
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t s) {
  g_call = {g, b, sh, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, hipStream_t* s) {
  *g = g_call.g;
  *b = g_call.b;
  *sh = g_call.sh;
  *s = g_call.s;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* stub, dim3 g, dim3 b, void**, size_t sh, hipStream_t) {
  const std::string& name = g_kernels[stub];
  if (!g_fail.empty() && name.find(g_fail) != std::string::npos) {
    g_fail.clear();
    g_log += "failed " + name + "\n";
    return result(hipErrorOutOfMemory);
  }
  // what the device refuses
  if (!g.x || !g.y || !g.z || g.y > 65535 || g.z > 65535 || b.x * b.y * b.z > 1024 ||
      sh > 160 * 1024)
    return result(hipErrorInvalidConfiguration);
  for (const auto& c : g_cost)
    if (name.find(c.first) != std::string::npos) g_clock += c.second;
  g_clock += 1e-3;
  g_log += name + "\n";
  return hipSuccess;
}

// ---- devices and errors
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  p->totalGlobalMem = size_t(288) << 30;
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "an error"; }
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}

// ---- memory
hipError_t hipMalloc(void** p, size_t n) {
  *p = std::calloc(1, n ? n : 1);
  return *p ? hipSuccess : result(hipErrorOutOfMemory);
}
hipError_t hipFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipGetSymbolAddress(void** p, const void* var) {
  *p = g_vars[var];
  return *p ? hipSuccess : result(hipErrorInvalidSymbol);
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  g_log += "copy\n";
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  std::memset(d, v, n);
  return hipSuccess;
}

// ---- streams, events, graphs
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t) new char;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  delete (char*)s;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  g_log += "wait\n";
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = (hipGraph_t) new char;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *e = (hipGraphExec_t) new char;
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  delete (char*)g;
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  delete (char*)e;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
  g_log += "graph\n";
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = (hipEvent_t) new Event;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
  delete (Event*)e;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  ((Event*)e)->at = g_clock;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
  *ms = (float)(((Event*)b)->at - ((Event*)a)->at);
  return hipSuccess;
}

}  // extern "C"
