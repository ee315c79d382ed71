// A stand-in for the HIP runtime with two devices, for tests on the CPU: device
// memory is host memory, kernels do nothing, and every operation on a stream is
// checked against the devices its memory and events belong to.  Load it with
// RTLD_GLOBAL before the library, whose calls then come here.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

namespace {
thread_local int cur = 0;
std::mutex mu;
std::map<const char*, std::pair<size_t, int>> blocks;  // base -> size, device
int violations = 0;

struct Stream { int dev; };
struct Event { int dev; };

int device_of(const void* p) {  // -1: host memory
  std::lock_guard<std::mutex> lk(mu);
  auto it = blocks.upper_bound(static_cast<const char*>(p));
  if (it == blocks.begin()) return -1;
  --it;
  return static_cast<const char*>(p) < it->first + it->second.first ? it->second.second : -1;
}
hipError_t foreign(const char* what, int want, int got) {
  std::fprintf(stderr, "%s: stream of device %d, object of device %d\n", what, want, got);
  std::lock_guard<std::mutex> lk(mu);
  ++violations;
  return hipErrorInvalidHandle;
}
hipError_t check(const char* what, hipStream_t s, const void* p) {
  const int want = s ? reinterpret_cast<Stream*>(s)->dev : cur, got = device_of(p);
  return got >= 0 && got != want ? foreign(what, want, got) : hipSuccess;
}
}  // namespace

extern "C" {
int two_devices_violations() { return violations; }

hipError_t hipGetDevice(int* d) { *d = cur; return hipSuccess; }
hipError_t hipSetDevice(int d) { return d == 0 || d == 1 ? (cur = d, hipSuccess) : hipErrorInvalidDevice; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
  *p = std::calloc(n, 1);
  std::lock_guard<std::mutex> lk(mu);
  blocks[static_cast<char*>(*p)] = {n, cur};
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lk(mu);
  blocks.erase(static_cast<char*>(p));
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return (*p = std::calloc(n, 1)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
  std::memcpy(d, s, n);
  const hipError_t e = check("copy to", st, d);
  return e ? e : check("copy from", st, s);
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t st) {
  std::memset(d, v, n);
  return check("memset", st, d);
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(new Stream{cur});
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { delete reinterpret_cast<Stream*>(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) { *d = s ? reinterpret_cast<Stream*>(s)->dev : cur; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(new Event{cur});
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<Event*>(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  const int want = s ? reinterpret_cast<Stream*>(s)->dev : cur, got = reinterpret_cast<Event*>(e)->dev;
  return want == got ? hipSuccess : foreign("event", want, got);
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
}
