// Shared host helpers: error reporting macros and an owning device buffer.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/xrtailor_amd.h"

namespace xrt {

void SetError(const std::string& msg);

#define XRT_CHECK_HIP(expr)                                                       \
  do {                                                                            \
    hipError_t _e = (expr);                                                       \
    if (_e != hipSuccess) {                                                       \
      ::xrt::SetError(std::string(#expr) + ": " + hipGetErrorString(_e));        \
      return XRT_ERR_HIP;                                                         \
    }                                                                             \
  } while (0)

#define XRT_REQUIRE(cond, code, msg) \
  do {                               \
    if (!(cond)) {                   \
      ::xrt::SetError(msg);          \
      return (code);                 \
    }                                \
  } while (0)

template <typename T>
struct DevBuf {
  T* ptr = nullptr;
  size_t n = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf() { Free(); }
  void Free() {
    if (ptr) (void)hipFree(ptr);
    ptr = nullptr;
    n = 0;
  }
  // n is count only when the memory is there: callers that keep a buffer of the right n must not
  // take a null one for it after a failure
  hipError_t Alloc(size_t count) {
    Free();
    if (count == 0) return hipSuccess;
    const hipError_t e = hipMalloc(reinterpret_cast<void**>(&ptr), count * sizeof(T));
    if (e == hipSuccess) {
      n = count;
    } else {
      ptr = nullptr;
      (void)hipGetLastError();  // else the next launch would report it again
    }
    return e;
  }
  // The copy has completed when this returns: callers upload from temporaries (set-up
  // vectors that die at the end of their scope), and HIP does not promise that an
  // asynchronous copy from pageable memory has read its source when the call returns
  // (the runtime may queue it to a worker thread). Never called under stream capture.
  hipError_t Upload(const T* host, size_t count, hipStream_t s) {
    if (count == 0) return hipSuccess;
    hipError_t e = hipMemcpyAsync(ptr, host, count * sizeof(T), hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return e;
    return hipStreamSynchronize(s);
  }
  hipError_t Upload(const std::vector<T>& host, hipStream_t s) {
    hipError_t e = Alloc(host.size());
    if (e != hipSuccess) return e;
    return Upload(host.data(), host.size(), s);
  }
};

}  // namespace xrt
