// A HIP runtime of plain host memory for the CPU tests of host code that
// orders copies and launches (test_copies.py).  A stream's work runs in order,
// either as soon as it is enqueued (eager) or not before the host waits for it
// (lazy), so that a missing wait shows as wrong bytes in one of the two; a
// closed gate in a stream stands for earlier work that is still running.
// Kernels run on the host, one thread after the other.
#pragma once

#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <condition_variable>
#include <deque>
#include <functional>
#include <memory>
#include <mutex>

#define __global__
struct dim3 {
  uint32_t x, y, z;
  dim3(uint32_t a = 1, uint32_t b = 1, uint32_t c = 1) : x(a), y(b), z(c) {}
};
struct uint4 {
  uint32_t x, y, z, w;
};
inline thread_local dim3 blockIdx, threadIdx, blockDim, gridDim;

typedef enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2,
               hipErrorInvalidHandle = 400 } hipError_t;
typedef enum { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 } hipMemcpyKind;
typedef int hipDevice_t;
constexpr unsigned hipHostMallocPortable = 1u, hipHostMallocCoherent = 0x40000000u;
constexpr unsigned hipEventDisableTiming = 2u, hipEventReleaseToSystem = 0x80000000u;
constexpr unsigned hipStreamNonBlocking = 1u;

namespace fake {
struct Gate {
  std::mutex mu;
  std::condition_variable cv;
  bool open = false;
  void pass() {
    std::unique_lock<std::mutex> lk(mu);
    cv.wait(lk, [&] { return open; });
  }
  void unlock() {
    std::lock_guard<std::mutex> lk(mu);
    open = true;
    cv.notify_all();
  }
};
struct Stream {
  int device = 0;
  std::recursive_mutex mu;
  std::deque<std::function<void()>> work;
  size_t enqueued = 0, ran = 0;
  bool gated = false;  // never run ahead of a wait
};
struct Event {
  int device = 0;
  unsigned flags = 0;
  Stream* stream = nullptr;
  size_t upto = 0;
};
inline bool eager = false;
inline thread_local int current = 0;
inline int devices = 1;
// what the code under test asked for
inline std::mutex log_mu;
inline size_t host_allocs = 0, transfers = 0;
inline unsigned host_flags = ~0u, event_flags = ~0u;  // and of all requests

inline void run(Stream* s, size_t upto) {
  std::lock_guard<std::recursive_mutex> lk(s->mu);
  while (s->ran < upto) {
    std::function<void()> f = std::move(s->work.front());
    s->work.pop_front();
    f();
    s->ran++;
  }
}
inline void enqueue(Stream* s, std::function<void()> f) {
  std::lock_guard<std::recursive_mutex> lk(s->mu);
  s->work.push_back(std::move(f));
  s->enqueued++;
  if (eager && !s->gated) run(s, s->enqueued);
}
inline void close_gate(Stream* s, Gate* g) {
  s->gated = true;
  enqueue(s, [g] { g->pass(); });
}
}  // namespace fake
typedef fake::Stream* hipStream_t;
typedef fake::Event* hipEvent_t;

inline const char* hipGetErrorString(hipError_t) { return "error"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { return *d = fake::current, hipSuccess; }
inline hipError_t hipSetDevice(int d) {
  if (d < 0 || d >= fake::devices) return hipErrorInvalidValue;
  return fake::current = d, hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) {
  std::lock_guard<std::mutex> lk(fake::log_mu);
  fake::host_allocs++;
  fake::host_flags &= flags;
  *p = aligned_alloc(4096, (n + 4095) / 4096 * 4096);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = new fake::Stream();
  (*s)->device = fake::current;
  return hipSuccess;
}
inline hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) {
  return *d = s->device, hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  size_t upto;
  {
    std::lock_guard<std::recursive_mutex> lk(s->mu);
    upto = s->enqueued;
  }
  return fake::run(s, upto), hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags) {
  *e = new fake::Event();
  (*e)->device = fake::current;
  (*e)->flags = flags;
  std::lock_guard<std::mutex> lk(fake::log_mu);
  fake::event_flags &= flags;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (e->device != s->device) return hipErrorInvalidHandle;
  e->stream = s;
  e->upto = s->enqueued;
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  if (e->stream) fake::run(e->stream, e->upto);
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind,
                                 hipStream_t s) {
  {
    std::lock_guard<std::mutex> lk(fake::log_mu);
    fake::transfers++;
  }
  fake::enqueue(s, [=] { memcpy(dst, src, n); });
  return hipSuccess;
}
template <typename F>
inline void fake_launch(dim3 grid, dim3 block, hipStream_t s, F f) {
  {
    std::lock_guard<std::mutex> lk(fake::log_mu);
    fake::transfers++;
  }
  fake::enqueue(s, [=] {
    gridDim = grid;
    blockDim = block;
    for (uint32_t b = 0; b < grid.x; b++)
      for (uint32_t t = 0; t < block.x; t++) {
        blockIdx = dim3(b);
        threadIdx = dim3(t);
        f();
      }
  });
}
#define hipLaunchKernelGGL(kernel, grid, block, shmem, stream, ...) \
  fake_launch(grid, block, stream, [=] { kernel(__VA_ARGS__); })
