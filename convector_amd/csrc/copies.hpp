// copies.hpp -- status helpers of the host code, and the copies between caller
// host memory and the device (copies.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

#include <string>

#include "../../include/convector.h"

namespace cvh {

// Records the message returned by cv_last_error() and passes the status on.
cv_status fail(cv_status s, const std::string& msg);
cv_status hip_fail(hipError_t e, const char* what);

// `rows` rows of `bytes` bytes of caller host memory and their place on the
// device.
struct CallerRect {
  void* host;
  void* dev;
  size_t bytes, rows, host_pitch, dev_pitch;
  // the rect before it ends where this one begins, in the same allocation: the
  // two share transfers
  bool follows;
  static CallerRect flat(const void* host, void* dev, size_t bytes, bool follows = false) {
    return CallerRect{const_cast<void*>(host), dev, bytes, 1, bytes, bytes, follows};
  }
};
// Copies between caller host memory and the device through pinned memory, a
// piece at a time, waiting for the copies (and so for the work queued before
// them on st): the runtime never copies from or to the caller's pageable
// memory, and nothing touches that memory after the call returns.
cv_status copy_caller_rects(const CallerRect* rects, size_t n, bool to_device, hipStream_t st);
cv_status copy_caller_memory(void* dst, const void* src, size_t bytes, bool to_device,
                             hipStream_t st);
// Downloads device memory that no queued work writes (a scene's tree) without
// waiting for the work of st, whose device it lies on.
cv_status copy_settled_rects(const CallerRect* rects, size_t n, hipStream_t st);

}  // namespace cvh

#define HIPTRY(x, what)                                        \
  do {                                                         \
    hipError_t e_ = (x);                                       \
    if (e_ != hipSuccess) return cvh::hip_fail(e_, what);      \
  } while (0)
