// copies.hip -- copies between caller host memory and the device, through
// pinned memory of the process.
#include <string.h>

#include <algorithm>
#include <condition_variable>
#include <mutex>
#include <new>
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

// What one piece of pinned memory takes: `rows` rows of `bytes` bytes on the
// device, packed in the piece, and the spans of host memory (from spans[first]
// on) whose bytes follow each other there.
struct Span {
  char* host;
  size_t bytes, rows, pitch;
};
struct Piece {
  char* dev;
  size_t bytes, rows, pitch, first, spans;
};
struct Plan {
  std::vector<Span> spans;
  std::vector<Piece> pieces;
  bool open = false;  // the last piece may take what follows it on the device

  void flat(char* host, char* dev, size_t n) {
    while (n) {
      Piece* last = open ? &pieces.back() : nullptr;
      if (last && (last->dev + last->bytes != dev || last->bytes == kPieceBytes)) last = nullptr;
      const size_t c = std::min(n, kPieceBytes - (last ? last->bytes : 0));
      if (last) {
        last->bytes += c;
        last->spans++;
      } else {
        pieces.push_back(Piece{dev, c, 1, 0, spans.size(), 1});
      }
      spans.push_back(Span{host, c, 1, 0});
      open = true;
      host += c;
      dev += c;
      n -= c;
    }
  }
  void add(const CallerRect& r) {
    if (!r.follows) open = false;
    if (!r.bytes || !r.rows) return;
    char *host = (char*)r.host, *dev = (char*)r.dev;
    const bool words = !((r.bytes | r.dev_pitch | (size_t)r.dev) & 15);
    if (r.rows == 1 || (r.host_pitch == r.bytes && r.dev_pitch == r.bytes)) {
      flat(host, dev, r.bytes * r.rows);
    } else if (r.bytes > kPieceBytes || !words) {
      // rows longer than a piece (an HDR rectangle from 43,691 pixels of width
      // on) or not of 16-byte words
      for (size_t y = 0; y < r.rows; y++) {
        open = false;
        flat(host + y * r.host_pitch, dev + y * r.dev_pitch, r.bytes);
      }
      open = false;
    } else {
      const size_t per = kPieceBytes / r.bytes;
      for (size_t y = 0; y < r.rows; y += per) {
        const size_t rows = std::min(per, r.rows - y);
        pieces.push_back(Piece{dev + y * r.dev_pitch, r.bytes, rows, r.dev_pitch, spans.size(), 1});
        spans.push_back(Span{host + y * r.host_pitch, r.bytes, rows, r.host_pitch});
      }
      open = false;
    }
  }
};

// settled: no queued work reads or writes the device memory, so that the copy
// runs on the ring's own stream, on the device of st.
cv_status copy_rects(const CallerRect* rects, size_t n, bool to_device, hipStream_t st,
                     bool settled) {
  Plan plan;
  try {
    for (size_t i = 0; i < n; i++) plan.add(rects[i]);
  } catch (const std::bad_alloc&) {
    return fail(CV_ERR_OUT_OF_MEMORY, "copy plan");
  }
  const std::vector<Piece>& ps = plan.pieces;
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
  auto host_copy = [&](size_t k) {
    char* b = pieces + (k % kPieces) * kPieceBytes;
    for (size_t j = 0; j < ps[k].spans; j++) {
      const Span& sp = plan.spans[ps[k].first + j];
      for (size_t y = 0; y < sp.rows; y++, b += sp.bytes) {
        char* h = sp.host + y * sp.pitch;
        if (to_device)
          memcpy(b, h, sp.bytes);
        else
          memcpy(h, b, sp.bytes);
      }
    }
  };
  auto dev_copy = [&](size_t k) -> cv_status {
    const Piece& p = ps[k];
    char* b = pieces + (k % kPieces) * kPieceBytes;
    const bool words = !((p.bytes | p.pitch | (size_t)p.dev) & 15);
    if (p.rows == 1 && (to_device || !words)) {
      HIPTRY(hipMemcpyAsync(to_device ? p.dev : b, to_device ? b : p.dev, p.bytes,
                            to_device ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, st),
             "copy");
    } else {
      const uint4* src = (const uint4*)(to_device ? b : p.dev);
      uint4* dst = (uint4*)(to_device ? p.dev : b);
      const size_t pk = p.bytes / 16, pitch = p.pitch / 16;
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
  const CallerRect r = to_device ? CallerRect::flat(src, dst, bytes)
                                 : CallerRect::flat(dst, const_cast<void*>(src), bytes);
  return copy_caller_rects(&r, 1, to_device, st);
}

}  // namespace cvh
