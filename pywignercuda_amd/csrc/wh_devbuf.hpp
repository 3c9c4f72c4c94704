// Device allocation owned by a plan.
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstddef>

namespace wh {

struct DeviceBuffer {
  void* p = nullptr;
  size_t bytes = 0;
  DeviceBuffer() = default;
  DeviceBuffer(const DeviceBuffer&) = delete;
  DeviceBuffer& operator=(const DeviceBuffer&) = delete;
  ~DeviceBuffer() {
    if (p) (void)hipFree(p);
  }
  // A new allocation of n bytes in place of the old one (contents are not kept).  On failure the
  // old one stays as it was: callers compare `bytes` with what a call needs, and kernels of the plan
  // may hold its address.
  hipError_t replace(size_t n) {
    void* q = nullptr;
    const hipError_t e = hipMalloc(&q, n ? n : 16);
    if (e != hipSuccess) return e;
    if (p) (void)hipFree(p);
    p = q;
    bytes = n;
    return hipSuccess;
  }
};

}  // namespace wh
