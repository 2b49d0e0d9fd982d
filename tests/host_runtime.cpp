// The HIP runtime calls that libsgeo.so makes, on host memory and without a
// GPU, for tests of the library's host side: "device" memory is calloc'ed
// within a limit, copies are memcpy, events and streams are empty.  Kernels do
// not run; their launches are recorded.  Errors behave as in ROCm 7:
// hipGetLastError returns the last failed call's code until it is read.
//
// Loaded with RTLD_GLOBAL before libsgeo.so, whose calls then resolve here.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace {

// never destroyed: the library's own exit still calls in here
std::mutex& mu = *new std::mutex;
auto& kernels = *new std::map<const void*, std::string>;  // host stub -> name
auto& blocks = *new std::map<void*, size_t>;              // device allocations
auto& log_ = *new std::string;  // one line per launch, allocation and free
auto& watch = *new std::string;
size_t used = 0, limit = SIZE_MAX, host_limit = SIZE_MAX;
int watch_arg = 0;
thread_local hipError_t last = hipSuccess;
thread_local struct {
  dim3 grid, block;
  size_t shmem;
  hipStream_t stream;
} config;

hipError_t error(hipError_t e) {
  if (e != hipSuccess) last = e;
  return e;
}

// bytes before each allocation, zero: the numbering's last-entry reads land
// here, since no kernel ran that would count its nodes
constexpr size_t PAD = 256;

}  // namespace

extern "C" {

// ---- test interface ----
void rt_limit(size_t bytes) { limit = bytes; }
void rt_host_limit(size_t bytes) { host_limit = bytes; }  // of one pinned allocation
size_t rt_used() { return used; }
void rt_clear() {
  std::lock_guard<std::mutex> l(mu);
  log_.clear();
}
const char* rt_log() { return log_.c_str(); }
// launches of kernels whose name holds `name` are logged with the pointer
// that is their argument `arg`
void rt_watch(const char* name, int arg) {
  watch = name;
  watch_arg = arg;
}

// ---- memory ----
hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> l(mu);
  if (used + n > limit) {
    log_ += "fail " + std::to_string(n) + "\n";
    return error(hipErrorOutOfMemory);
  }
  char* q = (char*)calloc(1, n + PAD);
  if (!q) return error(hipErrorOutOfMemory);
  *p = q + PAD;
  blocks[*p] = n;
  used += n;
  log_ += "malloc " + std::to_string(n) + "\n";
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  std::lock_guard<std::mutex> l(mu);
  auto it = blocks.find(p);
  if (it == blocks.end()) return error(hipErrorInvalidValue);
  used -= it->second;
  log_ += "free " + std::to_string(it->second) + "\n";
  blocks.erase(it);
  free((char*)p - PAD);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = n <= host_limit ? calloc(1, n) : nullptr;
  return *p ? hipSuccess : error(hipErrorOutOfMemory);
}
hipError_t hipHostFree(void* p) {
  free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  memset(d, v, n);
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static char scratch[1 << 16];
  *p = scratch;
  return hipSuccess;
}

// ---- device, streams, events ----
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
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
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  p->warpSize = 64;
  p->multiProcessorCount = 256;
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) {
  return e == hipErrorOutOfMemory ? "out of memory" : e == hipSuccess ? "no error" : "error";
}
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t)calloc(1, 8);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  free(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = (hipEvent_t)calloc(1, 8);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
  free(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
// every interval is shorter than the one before
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  static float t = 100.0f;
  *ms = t *= 0.9f;
  return hipSuccess;
}

// ---- graphs: not captured here (engines run with graphs off) ----
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  return error(hipErrorNotSupported);
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return error(hipErrorNotSupported); }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  return error(hipErrorNotSupported);
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return error(hipErrorNotSupported); }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

// ---- kernels ----
void** __hipRegisterFatBinary(const void*) {
  static void* module;
  return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* stub, char*, const char* name, unsigned, void*,
                           void*, void*, void*, int*) {
  kernels[stub] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t s) {
  config = {grid, block, shmem, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, hipStream_t* s) {
  *grid = config.grid;
  *block = config.block;
  *shmem = config.shmem;
  *s = config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* stub, dim3 grid, dim3 block, void** args, size_t,
                           hipStream_t) {
  std::lock_guard<std::mutex> l(mu);
  const std::string& name = kernels[stub];
  if (!grid.x || !grid.y || !grid.z || !block.x)
    return error(hipErrorInvalidConfiguration);
  // the one thing a kernel does here: started columns go on to iterate, as
  // after their first residual
  if (name.find("k_bpromote") != std::string::npos) {
    const int ncol = *(int*)args[0];
    int32_t* cst = *(int32_t**)args[1];
    for (int j = 0; j < ncol; j++)
      if (cst[j] == 1) cst[j] = 2;
  }
  log_ += "launch " + name;
  if (!watch.empty() && name.find(watch) != std::string::npos)
    log_ += " " + std::to_string((uintptr_t) * (void**)args[watch_arg]);
  log_ += "\n";
  return hipSuccess;
}

}  // extern "C"
