// Plain device copy, used to calibrate HBM byte counters (FETCH_SIZE and
// WRITE_SIZE of a copy of known size) and to write results to pinned memory; the
// staged transfers of the host-array entry points.
#include <algorithm>
#include <cstring>

#include "fe_internal.hpp"

namespace a2c {
namespace {
__global__ void k_copy_calib(const uint4* __restrict__ src, uint4* __restrict__ dst, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}
}  // namespace

hipError_t copy_to_pinned(hipStream_t st, void* pinned, const void* dsrc, size_t bytes) {
  const size_t n = (bytes + 15) / 16;
  if (n == 0) return hipSuccess;
  const int grid = (int)std::min<size_t>((n + 255) / 256, 512);
  hipLaunchKernelGGL(k_copy_calib, dim3(grid), dim3(256), 0, st, static_cast<const uint4*>(dsrc),
                     static_cast<uint4*>(pinned), n);
  return hipGetLastError();
}

namespace {
size_t part_size(size_t n, size_t parts, size_t min) {
  return std::max(min, ((n + parts - 1) / parts + 15) / 16 * 16);
}
}  // namespace

hipError_t HostTransfer::upload(hipStream_t st, char* stage, size_t cap, void* ddst, const void* src, size_t bytes) {
  for (size_t r = 0; r < bytes; r += cap) {
    if (r > 0)
      if (hipError_t e = hipStreamSynchronize(st)) return e;
    const size_t n = std::min(cap, bytes - r), part = part_size(n, PARTS, PART_MIN);
    for (size_t o = 0; o < n; o += part) {
      const size_t m = std::min(part, n - o);
      std::memcpy(stage + o, static_cast<const char*>(src) + r + o, m);
      if (hipError_t e = hipMemcpyAsync(static_cast<char*>(ddst) + r + o, stage + o, m, hipMemcpyHostToDevice, st))
        return e;
    }
  }
  return hipSuccess;
}

hipError_t HostTransfer::download(hipStream_t st, char* stage, size_t cap, void* dst, const void* dsrc, size_t bytes) {
  for (size_t r = 0; r < bytes; r += cap) {
    const size_t n = std::min(cap, bytes - r), part = part_size(n, PARTS, PART_MIN);
    int k = 0;
    for (size_t o = 0; o < n; o += part, ++k) {
      if (hipError_t e = copy_to_pinned(st, stage + o, static_cast<const char*>(dsrc) + r + o, std::min(part, n - o)))
        return e;
      if (o + part >= n) break;  // the last part is waited for with the stream
      if (!ev_[k]) {  // an event belongs to its stream's device
        hipDevice_t dev;
        if (hipError_t e = hipStreamGetDevice(st, &dev)) return e;
        const DeviceScope on(dev);
        if (hipError_t e = on.status()) return e;
        if (hipError_t e = hipEventCreateWithFlags(&ev_[k], hipEventDisableTiming)) return e;
      }
      if (hipError_t e = hipEventRecord(ev_[k], st)) return e;
    }
    k = 0;
    for (size_t o = 0; o < n; o += part, ++k) {
      if (hipError_t e = o + part < n ? hipEventSynchronize(ev_[k]) : hipStreamSynchronize(st)) return e;
      std::memcpy(static_cast<char*>(dst) + r + o, stage + o, std::min(part, n - o));
    }
  }
  return hipSuccess;
}

HostTransfer::~HostTransfer() {
  for (hipEvent_t e : ev_)
    if (e) (void)hipEventDestroy(e);
}
}  // namespace a2c

extern "C" int a2c_dev_copy(a2c_fe_ctx* c, void* dst, const void* src, size_t bytes) {
  if (!c) return A2C_EINVAL;
  c->err.clear();
  if (!dst || !src || (bytes & 15) || (((uintptr_t)dst | (uintptr_t)src) & 15))
    return a2c::set_err(c, A2C_EINVAL, "copy needs 16-byte aligned pointers and size");
  const size_t n = bytes / 16;
  if (n) {
    const int grid = (int)std::min<size_t>((n + 255) / 256, 8192);
    hipLaunchKernelGGL(a2c::k_copy_calib, dim3(grid), dim3(256), 0, c->stream, static_cast<const uint4*>(src),
                       static_cast<uint4*>(dst), n);
    A2C_HIP(c, hipGetLastError());
  }
  A2C_HIP(c, hipStreamSynchronize(c->stream));
  return A2C_OK;
}
