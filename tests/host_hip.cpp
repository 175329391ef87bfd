// A HIP runtime for tests of the library's host code where there is no GPU: kernels and copies do
// nothing and device memory reads as zero; what the library must wait for and what memory it
// holds is recorded.  Loaded into a process (RTLD_GLOBAL) before libflgpu.so, whose calls it takes.
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>

namespace {
std::mutex mu;
std::map<void *, size_t> blocks;
size_t live = 0, limit = (size_t)-1;
int nmalloc = 0;
std::set<void *> queued;  // executable graphs launched and not waited for
std::map<void *, std::set<void *>> marked;  // those that an event waits for
std::map<const void *, std::string> kernels;  // by their host stub: mangled name
std::map<std::string, int> launches;
int destroyed_in_flight = 0, graphs_destroyed = 0;
dim3 grid_, block_;
size_t shmem_;
hipStream_t stream_;
void idle() { queued.clear(); }
template <class T> T handle() { return (T)std::malloc(8); }
}  // namespace

extern "C" {

// for the tests
void host_hip_limit(size_t bytes) { limit = bytes; }
size_t host_hip_live() { return live; }
int host_hip_mallocs() { return nmalloc; }
int host_hip_destroyed_in_flight() { return destroyed_in_flight; }
int host_hip_graphs_destroyed() { return graphs_destroyed; }
int host_hip_launches(const char *part) {  // of kernels whose mangled name contains part
  int n = 0;
  for (auto &k : launches)
    if (k.first.find(part) != std::string::npos) n += k.second;
  return n;
}

hipError_t hipMalloc(void **p, size_t n) {
  std::lock_guard<std::mutex> g(mu);
  if (n > limit - live || live > limit) return hipErrorOutOfMemory;
  *p = std::calloc(1, n ? n : 1);
  blocks[*p] = n;
  live += n;
  nmalloc++;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  std::lock_guard<std::mutex> g(mu);
  if (!p) return hipSuccess;
  idle();  // waits for the device
  auto it = blocks.find(p);
  if (it == blocks.end()) return hipErrorInvalidValue;
  live -= it->second;
  blocks.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = std::calloc(1, n ? n : 1);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  std::free(p);
  return hipSuccess;
}
// what comes back from the device is zero, whatever went there
hipError_t hipMemcpyAsync(void *d, const void *, size_t n, hipMemcpyKind k, hipStream_t) {
  if (n && k == hipMemcpyDeviceToHost) std::memset(d, 0, n);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) {
  (void)hipMemcpyAsync(d, s, n, k, nullptr);
  std::lock_guard<std::mutex> g(mu);
  idle();
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
  *f = *t = (size_t)1 << 38;
  return hipSuccess;
}

hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  std::memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) {
  return e == hipErrorOutOfMemory ? "out of memory" : "error";
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
  *p = nullptr;
  return hipErrorInvalidValue;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = handle<hipStream_t>();
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  std::free((void *)s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  std::lock_guard<std::mutex> g(mu);
  idle();
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = handle<hipEvent_t>();
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
  std::free((void *)e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  std::lock_guard<std::mutex> g(mu);
  marked[(void *)e] = queued;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  std::lock_guard<std::mutex> g(mu);
  for (void *q : marked[(void *)e]) queued.erase(q);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float *t, hipEvent_t, hipEvent_t) {
  *t = 0.f;
  return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  *g = handle<hipGraph_t>();
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  std::free((void *)g);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  *e = handle<hipGraphExec_t>();
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
  std::lock_guard<std::mutex> g(mu);
  queued.insert((void *)e);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  std::lock_guard<std::mutex> g(mu);
  if (queued.erase((void *)e)) destroyed_in_flight++;
  graphs_destroyed++;
  std::free((void *)e);
  return hipSuccess;
}

hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t) {
  std::lock_guard<std::mutex> g(mu);
  launches[kernels[f]]++;
  return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t n, hipStream_t s) {
  grid_ = g;
  block_ = b;
  shmem_ = n;
  stream_ = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *n, hipStream_t *s) {
  *g = grid_;
  *b = block_;
  *n = shmem_;
  *s = stream_;
  return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { return (void **)&live; }
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *,
                           void *, dim3 *, dim3 *, int *) {
  kernels[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}

}  // extern "C"
