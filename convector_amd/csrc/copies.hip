// copies.hip -- copies between caller host memory and the device, through
// pinned memory of the process.
#include <string.h>

#include <algorithm>
#include <condition_variable>
#include <mutex>
#include <vector>

#include "copies.hpp"

namespace cvh {

namespace {
// Copies go through pinned memory in pieces, each with an event of its own, so
// that the host's copy of one piece overlaps the device's of the next (a
// 1280 x 736 bitmap and gbuffer, 7.5 MB: 10.2 ms by hipMemcpy2DAsync into
// pageable memory, row by row; 1.0 ms this way).  Coherent memory: kernels write
// the pieces and the host reads them after waiting for their events, which need
// not release to the system (without the flag, portable memory is not coherent).
constexpr size_t kPieceBytes = 2u << 20;
constexpr uint32_t kPieces = 8;
constexpr int kDevices = 64;

// The pieces of one copy at a time.  The process has kRings of them, so that
// threads copy at the same time; a ring's 16 MB are allocated when so many
// copies run at once for the first time (one copy after the other uses the
// first ring only), and kept until the process ends (freeing pinned memory at
// exit can run after the HIP runtime is torn down).
constexpr uint32_t kRings = 4;
struct Ring {
  bool leased = false;
  char* pieces = nullptr;
  // per device: an event is recorded on streams of its own device only
  hipEvent_t done[kDevices][kPieces] = {};
  hipStream_t stream[kDevices] = {};  // for copies that no queued work precedes
};
Ring g_rings[kRings];
std::mutex g_rings_mu;
// (never destroyed: a thread may still wait when the process exits)
std::condition_variable& g_ring_free = *new std::condition_variable;

// Leases a ring for a copy on st.  The last free one goes only to a copy whose
// stream has no earlier work left, so that copies behind a long launch never
// hold up one that can start.
class Lease {
 public:
  ~Lease() {
    if (!ring_) return;
    std::lock_guard<std::mutex> lk(g_rings_mu);
    ring_->leased = false;
    g_ring_free.notify_one();
  }
  cv_status take(hipStream_t st, bool ready) {
    std::unique_lock<std::mutex> lk(g_rings_mu);
    for (;;) {
      uint32_t free = 0;
      Ring* first = nullptr;
      for (Ring& r : g_rings) {
        if (r.leased) continue;
        if (!first) first = &r;
        free++;
      }
      if (free > (ready ? 0u : 1u)) {
        first->leased = true;
        ring_ = first;
        return CV_OK;
      }
      if (ready) {
        g_ring_free.wait(lk);
      } else {
        lk.unlock();
        HIPTRY(hipStreamSynchronize(st), "copy");
        ready = true;
        lk.lock();
      }
    }
  }
  // The ring with its memory, and its events on device dev (current).
  cv_status init(int dev) {
    if (!ring_->pieces)
      HIPTRY(hipHostMalloc((void**)&ring_->pieces, kPieceBytes * kPieces,
                           hipHostMallocPortable | hipHostMallocCoherent),
             "pinned alloc");
    for (hipEvent_t& e : ring_->done[dev])
      if (!e) HIPTRY(hipEventCreateWithFlags(&e, hipEventDisableTiming), "event");
    return CV_OK;
  }
  Ring* operator->() const { return ring_; }

 private:
  Ring* ring_ = nullptr;
};

// Makes the stream's device current while it lives: a copy works whatever
// device the calling thread has current (its events and launches belong to
// the stream's device).
struct OnDeviceOf {
  int device = 0, before = -1;
  cv_status enter(hipStream_t st) {
    int current = 0;
    HIPTRY(hipGetDevice(&current), "hipGetDevice");
    HIPTRY(hipStreamGetDevice(st, &device), "hipStreamGetDevice");
    if (device < 0 || device >= kDevices)
      return fail(CV_ERR_INVALID_ARGUMENT, "device index");
    if (device != current) {
      HIPTRY(hipSetDevice(device), "hipSetDevice");
      before = current;
    }
    return CV_OK;
  }
  ~OnDeviceOf() {
    if (before >= 0) (void)hipSetDevice(before);
  }
};

// Rows of `words` 16-byte words between a pitched and a packed buffer.
__global__ void k_copy_rows(const uint4* src, size_t spitch, uint4* dst, size_t dpitch,
                            uint32_t words, uint32_t rows) {
  for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < words * rows;
       k += gridDim.x * blockDim.x)
    dst[(size_t)(k / words) * dpitch + k % words] = src[(size_t)(k / words) * spitch + k % words];
}

// The part of a rect that one piece of pinned memory takes: rows
// [row, row + rows) of `bytes` bytes from byte `col` on.
struct Piece {
  const CallerRect* rc;
  size_t col, bytes, row, rows;
};

// settled: no queued work reads or writes the device memory, so that the copy
// runs on the ring's own stream, on the device of st.
cv_status copy_rects(const CallerRect* rects, size_t n, bool to_device, hipStream_t st,
                     bool settled) {
  std::vector<Piece> ps;
  for (size_t i = 0; i < n; i++) {
    const CallerRect& r = rects[i];
    if (!r.bytes || !r.rows) continue;
    const bool packed = r.rows == 1 || (r.host_pitch == r.bytes && r.dev_pitch == r.bytes);
    const bool words = !((r.bytes | r.dev_pitch | (size_t)r.dev) & 15);
    if (packed || r.bytes > kPieceBytes || !words) {
      // contiguous, or rows longer than a piece (an HDR rectangle from 43,691
      // pixels of width on) or not of 16-byte words: bytes of one row (or of
      // all)
      const size_t row_bytes = packed ? r.bytes * r.rows : r.bytes;
      for (size_t y = 0; y < (packed ? 1 : r.rows); y++)
        for (size_t c = 0; c < row_bytes; c += kPieceBytes)
          ps.push_back(Piece{&r, c, std::min(kPieceBytes, row_bytes - c), y, 1});
    } else {
      const size_t per = kPieceBytes / r.bytes;
      for (size_t y = 0; y < r.rows; y += per)
        ps.push_back(Piece{&r, 0, r.bytes, y, std::min(per, r.rows - y)});
    }
  }
  if (ps.empty()) return CV_OK;
  OnDeviceOf on;
  cv_status cs = on.enter(st);
  if (cs != CV_OK) return cs;
  Lease ring;
  if ((cs = ring.take(st, settled)) != CV_OK || (cs = ring.init(on.device)) != CV_OK) return cs;
  if (settled) {
    hipStream_t& own = ring->stream[on.device];
    if (!own) HIPTRY(hipStreamCreateWithFlags(&own, hipStreamNonBlocking), "hipStreamCreate");
    st = own;
  }
  char* const pieces = ring->pieces;
  hipEvent_t* const piece_done = ring->done[on.device];
  auto host_of = [](const Piece& p) { return (char*)p.rc->host + p.row * p.rc->host_pitch + p.col; };
  auto dev_of = [](const Piece& p) { return (char*)p.rc->dev + p.row * p.rc->dev_pitch + p.col; };
  auto host_copy = [&](size_t k) {
    const Piece& p = ps[k];
    char* b = pieces + (k % kPieces) * kPieceBytes;
    for (size_t y = 0; y < p.rows; y++) {
      char* h = host_of(p) + y * p.rc->host_pitch;
      if (to_device)
        memcpy(b + y * p.bytes, h, p.bytes);
      else
        memcpy(h, b + y * p.bytes, p.bytes);
    }
  };
  auto dev_copy = [&](size_t k) -> cv_status {
    const Piece& p = ps[k];
    char* b = pieces + (k % kPieces) * kPieceBytes;
    const bool words = !((p.bytes | p.rc->dev_pitch | (size_t)dev_of(p)) & 15);
    if (p.rows == 1 && (to_device || !words)) {
      HIPTRY(hipMemcpyAsync(to_device ? dev_of(p) : b, to_device ? b : dev_of(p), p.bytes,
                            to_device ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, st),
             "copy");
    } else {
      const uint4* src = (const uint4*)(to_device ? b : dev_of(p));
      uint4* dst = (uint4*)(to_device ? dev_of(p) : b);
      const size_t pk = p.bytes / 16, pitch = p.rc->dev_pitch / 16;
      const uint32_t blocks = (uint32_t)std::min<size_t>((pk * p.rows + 255) / 256, 256);
      hipLaunchKernelGGL(k_copy_rows, dim3(blocks), dim3(256), 0, st, src,
                         to_device ? pk : pitch, dst, to_device ? pitch : pk, (uint32_t)pk,
                         (uint32_t)p.rows);
      HIPTRY(hipGetLastError(), "copy");
    }
    HIPTRY(hipEventRecord(piece_done[k % kPieces], st), "event");
    return CV_OK;
  };
  hipError_t we = hipSuccess;
  if (to_device) {
    for (size_t k = 0; k < ps.size() && cs == CV_OK; k++) {
      if (k >= kPieces) we = hipEventSynchronize(piece_done[k % kPieces]);
      if (we != hipSuccess) break;
      host_copy(k);
      cs = dev_copy(k);
    }
  } else {
    size_t sent = 0;
    for (size_t k = 0; k < ps.size() && cs == CV_OK; k++) {
      while (sent < ps.size() && sent < k + kPieces && cs == CV_OK) cs = dev_copy(sent++);
      if (cs != CV_OK) break;
      we = hipEventSynchronize(piece_done[k % kPieces]);
      if (we != hipSuccess) break;
      host_copy(k);
    }
  }
  // the ring is the next caller's from here on
  const hipError_t se = hipStreamSynchronize(st);
  if (cs != CV_OK) return cs;
  HIPTRY(we, "copy");
  HIPTRY(se, "copy");
  return CV_OK;
}
}  // namespace

cv_status copy_caller_rects(const CallerRect* rects, size_t n, bool to_device, hipStream_t st) {
  return copy_rects(rects, n, to_device, st, false);
}

cv_status copy_settled_rects(const CallerRect* rects, size_t n, hipStream_t st) {
  return copy_rects(rects, n, false, st, true);
}

cv_status copy_caller_memory(void* dst, const void* src, size_t bytes, bool to_device,
                             hipStream_t st) {
  CallerRect r;
  r.host = to_device ? const_cast<void*>(src) : dst;
  r.dev = to_device ? dst : const_cast<void*>(src);
  r.bytes = r.host_pitch = r.dev_pitch = bytes;
  r.rows = 1;
  return copy_caller_rects(&r, 1, to_device, st);
}

}  // namespace cvh
