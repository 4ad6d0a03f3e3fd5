// copies.hip -- copies between caller host memory and the device, through
// pinned memory of the process.
#include <string.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "copies.hpp"

namespace cvh {

namespace {
// One pinned bounce buffer for the whole process, allocated on first use and
// kept until the process ends (freeing pinned memory at exit can run after
// the HIP runtime is torn down).  Copies go through it in pieces, each with
// an event of its own, so that the host's copy of one piece overlaps the
// device's of the next (a 1280 x 736 bitmap and gbuffer, 7.5 MB: 10.2 ms by
// hipMemcpy2DAsync into pageable memory, row by row; 1.0 ms this way).  Coherent
// memory: kernels write the pieces and the host reads them after waiting for
// their events, which need not release to the system (without the flag,
// portable memory is not coherent).
constexpr size_t kPieceBytes = 2u << 20;
constexpr uint32_t kPieces = 8;
constexpr int kBounceDevices = 64;
std::mutex g_bounce_mu;
char* g_bounce = nullptr;
// per device (an event is recorded on streams of its own device only)
hipEvent_t g_piece_done[kBounceDevices][kPieces] = {};

// Makes the stream's device current while it lives: a copy works whatever
// device the calling thread has current (its events and launches belong to
// the stream's device).
struct OnDeviceOf {
  int device = 0, before = -1;
  cv_status enter(hipStream_t st) {
    int current = 0;
    HIPTRY(hipGetDevice(&current), "hipGetDevice");
    HIPTRY(hipStreamGetDevice(st, &device), "hipStreamGetDevice");
    if (device < 0 || device >= kBounceDevices)
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

// The events of device dev (current), with the bounce buffer allocated;
// g_bounce_mu held.
cv_status bounce_init(int dev, hipEvent_t** done) {
  if (!g_bounce)
    HIPTRY(hipHostMalloc((void**)&g_bounce, kPieceBytes * kPieces,
                         hipHostMallocPortable | hipHostMallocCoherent),
           "pinned alloc");
  for (hipEvent_t& e : g_piece_done[dev])
    if (!e) HIPTRY(hipEventCreateWithFlags(&e, hipEventDisableTiming), "event");
  *done = g_piece_done[dev];
  return CV_OK;
}

// Rows of `words` 16-byte words between a pitched and a packed buffer.
__global__ void k_copy_rows(const uint4* src, size_t spitch, uint4* dst, size_t dpitch,
                            uint32_t words, uint32_t rows) {
  for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < words * rows;
       k += gridDim.x * blockDim.x)
    dst[(size_t)(k / words) * dpitch + k % words] = src[(size_t)(k / words) * spitch + k % words];
}

// The part of a rect that one piece of the bounce buffer takes: rows
// [row, row + rows) of `bytes` bytes from byte `col` on.
struct Piece {
  const CallerRect* rc;
  size_t col, bytes, row, rows;
};
}  // namespace

cv_status copy_caller_rects(const CallerRect* rects, size_t n, bool to_device, hipStream_t st) {
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
  std::lock_guard<std::mutex> lk(g_bounce_mu);
  hipEvent_t* piece_done = nullptr;
  cs = bounce_init(on.device, &piece_done);
  if (cs != CV_OK) return cs;
  auto host_of = [](const Piece& p) { return (char*)p.rc->host + p.row * p.rc->host_pitch + p.col; };
  auto dev_of = [](const Piece& p) { return (char*)p.rc->dev + p.row * p.rc->dev_pitch + p.col; };
  auto host_copy = [&](size_t k) {
    const Piece& p = ps[k];
    char* b = g_bounce + (k % kPieces) * kPieceBytes;
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
    char* b = g_bounce + (k % kPieces) * kPieceBytes;
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
  // the bounce buffer is the next caller's from here on
  const hipError_t se = hipStreamSynchronize(st);
  if (cs != CV_OK) return cs;
  HIPTRY(we, "copy");
  HIPTRY(se, "copy");
  return CV_OK;
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
