// A host-only stand-in for the HIP runtime calls of libminife_hip.so, for tests
// of the library's host code without a GPU.  Device memory is host memory (zeroed,
// at most `capacity` bytes in all), kernels are not run, and a stream only knows
// whether something has been launched on it that nobody has waited for.
#include <hip/hip_runtime_api.h>

#include <chrono>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

struct ihipStream_t {
  uint64_t launch = 0;  // clock of the last launch that is not known to be done; 0: none
  bool capturing = false;
};

namespace {
struct Alloc {
  size_t bytes;
  uint64_t birth;
};
std::recursive_mutex mu;
uint64_t tick = 0;
std::map<char*, Alloc> live;
std::vector<ihipStream_t*> streams;
size_t used = 0, capacity = size_t(1) << 30;
int free_delay_ms = 0;
long mallocs = 0, frees = 0, hazards = 0, foreign_waits = 0, capture_breaks = 0, host_fail = 0;
thread_local ihipStream_t* mine = nullptr;  // the stream of the context this thread works for

struct Config {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
};
thread_local std::vector<Config> configs;

void wait_all() {
  for (ihipStream_t* s : streams) s->launch = 0;
}
void launched(hipStream_t s) {
  std::lock_guard<std::recursive_mutex> lock(mu);
  if (s) s->launch = ++tick;
}
// Memory cleared on stream s that another stream's unfinished work may still use:
// the allocation was there when that work was launched.
void writes(void* p, hipStream_t s) {
  std::lock_guard<std::recursive_mutex> lock(mu);
  auto it = live.upper_bound(static_cast<char*>(p));
  if (it == live.begin()) return;
  --it;
  for (ihipStream_t* t : streams)
    if (t != s && t->launch > it->second.birth) ++hazards;
}
}  // namespace

extern "C" {

// ---- for the tests -------------------------------------------------------------
void stub_capacity(size_t bytes) { capacity = bytes; }
void stub_free_delay(int ms) { free_delay_ms = ms; }
size_t stub_used() { return used; }
long stub_mallocs() { return mallocs; }
long stub_frees() { return frees; }
long stub_hazards() { return hazards; }
long stub_foreign_waits() { return foreign_waits; }
long stub_capture_breaks() { return capture_breaks; }
void stub_host_fail(long n) { host_fail = n; }  // the n-th next pinned allocation fails
// This thread waits only for its own context's stream: the i-th one created.
void stub_thread_stream(int i) { mine = i < 0 ? nullptr : streams[(size_t)i]; }
void stub_begin_capture(int i) { streams[(size_t)i]->capturing = true; }
void stub_end_capture(int i) { streams[(size_t)i]->capturing = false; }

// ---- HIP -----------------------------------------------------------------------
void** __hipRegisterFatBinary(const void*) {
  static void* h = nullptr;
  return &h;
}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*,
                           void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
  configs.push_back(Config{grid, block, shared, stream});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
  const Config c = configs.back();
  configs.pop_back();
  *grid = c.grid;
  *block = c.block;
  *shared = c.shared;
  *stream = c.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t s) {
  launched(s);
  return hipSuccess;
}

hipError_t hipMalloc(void** out, size_t bytes) {
  std::lock_guard<std::recursive_mutex> lock(mu);
  if (used + bytes > capacity) return hipErrorOutOfMemory;
  char* p = static_cast<char*>(std::calloc(1, bytes ? bytes : 1));
  live[p] = Alloc{bytes, ++tick};
  used += bytes;
  ++mallocs;
  *out = p;
  return hipSuccess;
}
hipError_t hipFree(void* p) {  // waits for the whole device
  if (p && free_delay_ms > 0) std::this_thread::sleep_for(std::chrono::milliseconds(free_delay_ms));
  std::lock_guard<std::recursive_mutex> lock(mu);
  if (!p) return hipSuccess;
  auto it = live.find(static_cast<char*>(p));
  if (it == live.end()) return hipErrorInvalidValue;
  wait_all();
  used -= it->second.bytes;
  std::free(p);
  live.erase(it);
  ++frees;
  return hipSuccess;
}
hipError_t hipHostMalloc(void** out, size_t bytes, unsigned) {
  if (host_fail > 0 && --host_fail == 0) return hipErrorOutOfMemory;
  *out = std::calloc(1, bytes ? bytes : 1);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* free_b, size_t* total) {
  std::lock_guard<std::recursive_mutex> lock(mu);
  *free_b = capacity - used;
  *total = capacity;
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t st) {
  if (kind != hipMemcpyDeviceToHost) writes(d, st);
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t st) {
  writes(d, st);
  std::memset(d, v, n);
  launched(st);
  return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  std::lock_guard<std::recursive_mutex> lock(mu);
  *s = new ihipStream_t();
  streams.push_back(*s);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  std::lock_guard<std::recursive_mutex> lock(mu);
  if (s->capturing) {
    ++capture_breaks;
    return hipErrorStreamCaptureUnsupported;
  }
  if (mine && s != mine) ++foreign_waits;
  s->launch = 0;
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
  s->capturing = true;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
  s->capturing = false;
  *g = reinterpret_cast<hipGraph_t>(s);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
  *e = reinterpret_cast<hipGraphExec_t>(g);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) {
  launched(s);
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

hipError_t hipEventCreate(hipEvent_t* e) {
  static int dummy;
  *e = reinterpret_cast<hipEvent_t>(&dummy);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1.0f;
  return hipSuccess;
}

hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(static_cast<void*>(p), 0, sizeof(*p));
  p->multiProcessorCount = 256;
  p->totalGlobalMem = capacity;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 100000;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 4;
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
  std::memset(static_cast<void*>(a), 0, sizeof(*a));
  a->type = hipMemoryTypeDevice;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static char scratch[1 << 20];
  *p = scratch;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub"; }

}  // extern "C"
