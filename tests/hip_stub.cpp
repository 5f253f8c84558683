// A HIP runtime without a GPU, for tests of the library's host code: device
// memory is host memory set to zero, a kernel launch runs nothing and is noted
// down, and the caller chooses which allocation fails.  Loaded before the
// library with its symbols global, so the library's calls bind to it
// (tests/hip_stub.py).
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <vector>

namespace {

struct Launch {
  std::string kernel;
  dim3 grid, block;
  void* first;  // first eight bytes of the arguments
};

// What a kernel would have written: `bytes` to the memory its argument `arg`
// points to.
struct Effect {
  std::string part;
  int arg;
  std::vector<char> bytes;
};

std::mutex lock;
std::vector<Effect> effects;
std::map<const void*, std::string> names;
std::vector<Launch> launches;
std::set<void*> live;
long fail_in = 0, allocations = 0;
size_t free_bytes = size_t(1) << 37;
struct Config {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
};
std::vector<Config> configs;
hipError_t last = hipSuccess;

}  // namespace

extern "C" {

// ---- for the test ----

// the k-th hipMalloc from now fails (0: none)
void stub_fail_in(long k) { fail_in = k; }
long stub_allocations() { return allocations; }
long stub_live() { return (long)live.size(); }
void stub_clear_launches() { launches.clear(); }
// launches of kernels whose name holds `part` write n bytes to the memory that
// their argument `arg` points to
void stub_effect(const char* part, int arg, const char* bytes, size_t n) {
  effects.push_back({part, arg, std::vector<char>(bytes, bytes + n)});
}
// launches of kernels whose name holds `part`; null_first: only those whose
// first argument is a null pointer; over: only those of more work-items
long stub_launches(const char* part, int null_first, unsigned long long over) {
  long n = 0;
  for (const Launch& l : launches)
    if (l.kernel.find(part) != std::string::npos &&
        (!null_first || !l.first) &&
        (unsigned long long)l.grid.x * l.grid.y * l.grid.z * l.block.x *
                l.block.y * l.block.z > over)
      ++n;
  return n;
}
// work-items over all launches of kernels whose name holds `part`
unsigned long long stub_work_items(const char* part) {
  unsigned long long n = 0;
  for (const Launch& l : launches)
    if (l.kernel.find(part) != std::string::npos)
      n += (unsigned long long)l.grid.x * l.grid.y * l.grid.z * l.block.x *
           l.block.y * l.block.z;
  return n;
}

// ---- the runtime ----

void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name,
                           unsigned, void*, void*, dim3*, dim3*, int*) {
  names[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds,
                                      hipStream_t stream) {
  configs.push_back({grid, block, lds, stream});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds,
                                     hipStream_t* stream) {
  const Config c = configs.back();
  configs.pop_back();
  *grid = c.grid;
  *block = c.block;
  *lds = c.lds;
  *stream = c.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args,
                           size_t, hipStream_t) {
  std::lock_guard<std::mutex> hold(lock);
  Launch l{names.count(f) ? names[f] : "?", grid, block, nullptr};
  std::memcpy(&l.first, args[0], sizeof(void*));
  launches.push_back(l);
  for (const Effect& e : effects)
    if (l.kernel.find(e.part) != std::string::npos)
      std::memcpy(*static_cast<void**>(args[e.arg]), e.bytes.data(),
                  e.bytes.size());
  return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t bytes) {
  std::lock_guard<std::mutex> hold(lock);
  ++allocations;
  if (fail_in > 0 && --fail_in == 0) {
    *p = nullptr;
    return last = hipErrorOutOfMemory;
  }
  *p = std::calloc(bytes ? bytes : 1, 1);
  if (!*p) return last = hipErrorOutOfMemory;
  live.insert(*p);
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> hold(lock);
  if (p && !live.erase(p)) {
    std::fprintf(stderr, "hipFree of a pointer that is not allocated\n");
    std::abort();
  }
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  *p = std::calloc(bytes ? bytes : 1, 1);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind,
                          hipStream_t) {
  std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* free, size_t* total) {
  *free = free_bytes;
  *total = size_t(288) << 30;
  return hipSuccess;
}

hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) {
  return e == hipErrorOutOfMemory ? "out of memory" : "error";
}
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  switch (a) {
    case hipDeviceAttributeWarpSize: *v = 64; break;
    case hipDeviceAttributeMultiprocessorCount: *v = 256; break;
    case hipDeviceAttributeMaxThreadsPerBlock: *v = 1024; break;
    case hipDeviceAttributeMaxSharedMemoryPerBlock: *v = 65536; break;
    case hipDeviceAttributeMaxGridDimX: *v = 0x7fffffff; break;
    default: *v = 2048; break;
  }
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->name, "stub");
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  p->maxThreadsPerBlock = 1024;
  return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) {
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* symbol) {
  *p = const_cast<void*>(symbol);
  return hipSuccess;
}

hipError_t hipStreamCreate(hipStream_t* s) {
  *s = (hipStream_t)8;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t)8;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) {
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = (hipGraph_t)8;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*,
                               char*, size_t) {
  *e = (hipGraphExec_t)8;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = (hipEvent_t)8;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = (hipEvent_t)8;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1.0f;
  return hipSuccess;
}

}  // extern "C"
