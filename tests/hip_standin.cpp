// A host-only stand-in for the HIP runtime with two devices, for tests of the
// library's host code without a GPU: device memory is host memory, copies
// happen at once, kernels do nothing.  As in HIP, a stream and an event belong
// to the device that was current when they were created, and an event can only
// be recorded on a stream of its own device.  Freeing host memory that is not
// allocated ends the program.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <set>

namespace {
thread_local int current = 0;
struct Owned {
  int device;
};
int device_of(hipStream_t s) { return s ? reinterpret_cast<Owned *>(s)->device : current; }
// never destroyed: used until the process ends
std::mutex &host_mu = *new std::mutex;
std::set<void *> &host = *new std::set<void *>;
alignas(256) double symbol[(1 << 18) + 32];
}  // namespace

extern "C" {
hipError_t hipGetDevice(int *d) {
  *d = current;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  if (d < 0 || d > 1) return hipErrorInvalidDevice;
  current = d;
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
  *p = std::malloc(n);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  if (std::getenv("STANDIN_NO_PINNED_MEMORY")) return hipErrorOutOfMemory;
  const hipError_t e = hipMalloc(p, n);
  std::lock_guard<std::mutex> lock(host_mu);
  if (e == hipSuccess) host.insert(*p);
  return e;
}
hipError_t hipHostFree(void *p) {
  std::lock_guard<std::mutex> lock(host_mu);
  if (!host.erase(p)) {
    std::fprintf(stderr, "hipHostFree of memory that is not allocated\n");
    std::_Exit(3);
  }
  return hipFree(p);
}
hipError_t hipMemset(void *p, int v, size_t n) {
  std::memset(p, v, n);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) {
  return hipMemcpy(d, s, n, k);
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(new Owned{current});
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  delete reinterpret_cast<Owned *>(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(new Owned{current});
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
  delete reinterpret_cast<Owned *>(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  return reinterpret_cast<Owned *>(e)->device == device_of(s) ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 1;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorInvalidHandle ? "invalid handle" : "error"; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
  *p = symbol;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
}
