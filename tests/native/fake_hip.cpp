// A HIP runtime on host memory for the tests of the drivers' host code: it
// counts the streams, events and buffers that are live, keeps device memory
// within a limit and lets any call fail.  Kernels are not run, except that the
// check of a request order is done on the host.  Built as libamdhip64.so.7 and
// found through LD_LIBRARY_PATH, it takes the runtime's place for the library
// under test; streams do everything at once.
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <vector>

#include <hip/hip_runtime_api.h>

namespace {

std::mutex mu;
std::set<void*> streams, events, graphs, execs;
std::map<void*, size_t> buffers, uncached;
std::map<const void*, std::string> kernels;
size_t limit = ~(size_t)0, used = 0;
long calls = 0, fail_at = 0, wrong = 0;
hipError_t last = hipSuccess;

// every call that can fail passes here: call number fail_at fails
bool fails() { return ++calls == fail_at; }
#define GATE                                  \
  std::lock_guard<std::mutex> g_(mu);         \
  if (fails()) return last = hipErrorUnknown;

void* token(std::set<void*>& s) {
  void* p = std::malloc(16);
  s.insert(p);
  return p;
}
hipError_t drop(std::set<void*>& s, void* p) {
  if (!s.erase(p)) {
    ++wrong;  // never created, or destroyed already
    return hipErrorInvalidValue;
  }
  std::free(p);
  return hipSuccess;
}
hipError_t allocate(void** p, size_t n) {
  if (n > limit - used || used > limit) return last = hipErrorOutOfMemory;
  *p = std::calloc(1, n ? n : 1);
  buffers[*p] = n;
  used += n;
  return hipSuccess;
}

template <class T>
T arg(void** args, int i) {
  return *(T*)args[i];
}

}  // namespace

extern "C" {

// what the test reads and sets
long fake_live(int what) {
  std::lock_guard<std::mutex> g(mu);
  switch (what) {
    case 0: return (long)streams.size();
    case 1: return (long)events.size();
    case 2: return (long)buffers.size();
    case 3: return (long)graphs.size() + (long)execs.size();
    case 4: return wrong;
    case 5: return calls;
    default: return (long)used;
  }
}
void fake_fail_at(long n) {
  std::lock_guard<std::mutex> g(mu);
  calls = 0;
  fail_at = n;
}
void fake_limit(size_t n) { limit = n; }

hipError_t hipMalloc(void** p, size_t n) {
  GATE return allocate(p, n);
}
hipError_t hipExtMallocWithFlags(void** p, size_t n, unsigned) {
  GATE* p = std::malloc(16);  // the arena: never touched by host code
  uncached[*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> g(mu);
  if (!p) return hipSuccess;
  auto it = buffers.find(p);
  if (it == buffers.end()) {
    ++wrong;
    return hipErrorInvalidValue;
  }
  used -= it->second;
  buffers.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  GATE std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  GATE std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) {
  GATE std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  GATE std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemcpyToSymbol(const void*, const void*, size_t, size_t, hipMemcpyKind) {
  GATE return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static char block[1 << 16];
  GATE* p = block;
  return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t* s) {
  GATE* s = (hipStream_t)token(streams);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  std::lock_guard<std::mutex> g(mu);
  return drop(streams, s);
}
hipError_t hipStreamSynchronize(hipStream_t) { GATE return hipSuccess; }
hipError_t hipDeviceSynchronize() { GATE return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  GATE* e = (hipEvent_t)token(events);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  std::lock_guard<std::mutex> g(mu);
  return drop(events, e);
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { GATE return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { GATE return hipSuccess; }
hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t) {
  GATE* t = 1.0f;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { GATE return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* gr) {
  GATE* gr = (hipGraph_t)token(graphs);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  GATE* e = (hipGraphExec_t)token(execs);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { GATE return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t gr) {
  std::lock_guard<std::mutex> g(mu);
  return drop(graphs, gr);
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  std::lock_guard<std::mutex> g(mu);
  return drop(execs, e);
}
hipError_t hipGetDevice(int* d) {
  GATE* d = 0;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  GATE* v = a == hipDeviceAttributeWallClockRate ? 100000 : 256;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  GATE std::memset(p, 0, sizeof *p);
  p->totalGlobalMem = 288ull << 30;
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetLastError() {
  std::lock_guard<std::mutex> g(mu);
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "failed on purpose"; }

hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) {
  GATE
  // list_order_k(order, total, inv, lost): counts the places that did not survive
  if (kernels[f].find("list_order_k") != std::string::npos) {
    const unsigned* order = arg<const unsigned*>(args, 0);
    const unsigned long long total = arg<unsigned long long>(args, 1);
    std::vector<bool> seen(total, false);
    for (unsigned long long k = 0; k < total; ++k) {
      if (order[k] >= total || seen[order[k]]) ++*arg<unsigned long long*>(args, 3);
      else seen[order[k]] = true;
    }
  }
  return hipSuccess;
}

void** __hipRegisterFatBinary(const void*) {
  static void* h;
  return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  kernels[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
  *g = dim3(1);
  *b = dim3(1);
  *m = 0;
  *s = nullptr;
  return hipSuccess;
}

}  // extern "C"
