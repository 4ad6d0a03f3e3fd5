// Checks of convector_amd/csrc/copies.hip on a HIP runtime of plain host
// memory: copies_check NAME runs one of them (test_copies.py).
#include "../convector_amd/csrc/copies.hip"

#include <stdio.h>
#include <unistd.h>

#include <chrono>
#include <future>

namespace cvh {
cv_status fail(cv_status s, const std::string&) { return s; }
cv_status hip_fail(hipError_t, const char*) { return CV_ERR_DEVICE; }
}  // namespace cvh

using cvh::CallerRect;

#define CHECK(x)                                             \
  do {                                                       \
    if (!(x)) {                                              \
      printf("line %d: %s\n", __LINE__, #x);                 \
      exit(1);                                               \
    }                                                        \
  } while (0)

constexpr size_t P = cvh::kPieceBytes;

hipStream_t new_stream() {
  hipStream_t s;
  hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
  return s;
}

// One rect of a call: rows of bytes, host and device pitch, and the device
// memory's offset from a 16-byte boundary.
struct Shape {
  size_t bytes, rows, host_pitch, dev_pitch, dev_off;
};

// Rects of the shapes in one call, there and back: the rects' bytes arrive, and
// every byte between and around them stays as it was.
void copy_shapes(const std::vector<Shape>& shapes, hipStream_t st) {
  constexpr size_t kEdge = 64;
  struct Mem {
    std::vector<char> host, before;
    char* dev;
    size_t host_n, dev_n;
  };
  for (bool up : {true, false}) {
    std::vector<Mem> mem(shapes.size());
    std::vector<CallerRect> rects;
    for (size_t i = 0; i < shapes.size(); i++) {
      const Shape& s = shapes[i];
      Mem& m = mem[i];
      m.host_n = s.rows ? (s.rows - 1) * s.host_pitch + s.bytes : 0;
      m.dev_n = s.rows ? (s.rows - 1) * s.dev_pitch + s.bytes : 0;
      m.host.resize(m.host_n + 2 * kEdge);
      const size_t n = m.dev_n + s.dev_off + 2 * kEdge;
      m.dev = (char*)aligned_alloc(16, (n + 15) / 16 * 16);
      for (size_t k = 0; k < m.host.size(); k++) m.host[k] = (char)(k * 7 + i);
      for (size_t k = 0; k < n; k++) m.dev[k] = (char)(k * 13 + (k >> 8) + 5 * i + 101);
      if (up)
        m.before.assign(m.dev, m.dev + n);
      else
        m.before = m.host;
      rects.push_back(CallerRect{m.host.data() + kEdge, m.dev + kEdge + s.dev_off, s.bytes, s.rows,
                                 s.host_pitch, s.dev_pitch, false});
    }
    CHECK(cvh::copy_caller_rects(rects.data(), rects.size(), up, st) == CV_OK);
    for (size_t i = 0; i < shapes.size(); i++) {
      const Shape& s = shapes[i];
      Mem& m = mem[i];
      char* host = m.host.data() + kEdge;
      char* dev = m.dev + kEdge + s.dev_off;
      char* dst = up ? dev : host;
      const char* src = up ? host : dev;
      const size_t dp = up ? s.dev_pitch : s.host_pitch, sp = up ? s.host_pitch : s.dev_pitch;
      std::vector<char> want = m.before;
      for (size_t y = 0; y < s.rows; y++)
        memcpy(want.data() + kEdge + (up ? s.dev_off : 0) + y * dp, src + y * sp, s.bytes);
      const char* all = up ? m.dev : m.host.data();
      CHECK(memcmp(all, want.data(), want.size()) == 0);
      CHECK(memcmp(dst, src, s.rows ? s.bytes : 0) == 0);
    }
    for (Mem& m : mem) free(m.dev);
  }
}

// Pieces and their boundaries: flat copies around one piece and around all
// pieces of the buffer, pitched rects of part of a piece, of several, with one
// row more than a piece takes, with rows that are no 16-byte words or longer
// than a piece, and several rects in one call.
void check_shapes() {
  for (bool eager : {false, true}) {
    fake::eager = eager;
    hipStream_t st = new_stream();
    for (size_t n : {size_t(1), size_t(15), size_t(16), size_t(17), P - 1, P, P + 1, 8 * P - 1, 8 * P,
                     8 * P + 1, 9 * P + 5, 17 * P + 16})
      for (size_t off : {0, 4}) copy_shapes({{n, 1, n, n, off}}, st);
    const size_t per = P / 1024;  // rows of 1024 bytes in a piece
    for (size_t rows : {size_t(1), size_t(2), per - 1, per, per + 1, 8 * per, 8 * per + 1, 9 * per + 3})
      copy_shapes({{1024, rows, 1040, 1536, 0}}, st);
    copy_shapes({{1000, 5, 1000, 1008, 0}, {1024, 5, 1024, 1032, 0}, {1024, 5, 1030, 1024, 8}}, st);
    copy_shapes({{P + 48, 3, P + 64, P + 4096, 0}, {3 * P, 2, 3 * P, 3 * P, 0}}, st);
    copy_shapes({{64, 3, 100, 128, 0}, {0, 5, 16, 16, 0}, {16, 0, 16, 16, 0}, {5 * P + 3, 1, 0, 0, 0},
                 {4096, 4 * P / 4096, 4096, 8192, 0}, {7, 1, 7, 7, 3}}, st);
  }
}

// Kernels write the pinned pieces and the host reads them after waiting for an
// event: the memory is coherent, or the events release to the system.
void check_coherent() {
  copy_shapes({{1024, 4, 1024, 2048, 0}}, new_stream());
  CHECK((fake::host_flags & hipHostMallocCoherent) || (fake::event_flags & hipEventReleaseToSystem));
}

// A copy works whatever device the calling thread has current, with events of
// the stream's device, and leaves the current device as it was.
void check_devices() {
  fake::devices = 3;
  for (int on : {2, 0, 1}) {
    fake::current = on;
    hipStream_t st = new_stream();
    for (int current : {0, 1, 2}) {
      fake::current = current;
      copy_shapes({{1024, 4, 1024, 2048, 0}, {3 * P, 1, 0, 0, 0}}, st);
      CHECK(fake::current == current);
    }
  }
}

// Copies that wait for earlier work of their streams do not hold up those that
// can start at once, however many they are; the pinned memory stays bounded.
void check_threads() {
  std::vector<char> dev(3 * P + 5, 'd');
  std::vector<std::vector<char>> host(8, std::vector<char>(dev.size()));
  fake::Gate gate;
  std::vector<std::future<cv_status>> waiting;
  auto download = [&](size_t k, hipStream_t st) {
    return cvh::copy_caller_memory(host[k].data(), dev.data(), dev.size(), false, st);
  };
  for (size_t k = 0; k < 6; k++) {
    hipStream_t st = new_stream();
    fake::close_gate(st, &gate);
    waiting.push_back(std::async(std::launch::async, download, k, st));
  }
  for (auto& w : waiting)
    CHECK(w.wait_for(std::chrono::milliseconds(200)) == std::future_status::timeout);
  for (size_t k = 6; k < 8; k++) {
    auto free_one = std::async(std::launch::async, download, k, new_stream());
    const bool done = free_one.wait_for(std::chrono::seconds(10)) == std::future_status::ready;
    if (!done) {
      printf("a copy waits for the work of other streams\n");
      fflush(stdout);
      _exit(1);
    }
    CHECK(free_one.get() == CV_OK && host[k] == dev);
  }
  gate.unlock();
  for (size_t k = 0; k < 6; k++) CHECK(waiting[k].get() == CV_OK && host[k] == dev);
  CHECK(fake::host_allocs <= 4);
}

// Many threads at once, each with a stream of its own: every copy arrives.
void check_crowd() {
  std::vector<std::future<void>> all;
  for (int t = 0; t < 12; t++)
    all.push_back(std::async(std::launch::async, [] {
      hipStream_t st = new_stream();
      for (int k = 0; k < 3; k++)
        copy_shapes({{1024, 700, 1040, 1536, 0}, {P + 9, 1, 0, 0, 4}}, st);
    }));
  for (auto& a : all) a.get();
  CHECK(fake::host_allocs <= 4);
}

// Device memory that no queued work writes is copied without waiting for the
// object's stream.
void check_settled() {
  fake::devices = 2;
  fake::current = 1;
  hipStream_t st = new_stream();
  fake::current = 0;
  fake::Gate gate;
  fake::close_gate(st, &gate);
  std::vector<char> dev(3 * P + 5, 'd'), host(dev.size());
  const CallerRect r = CallerRect::flat(host.data(), dev.data(), dev.size());
  auto copy = std::async(std::launch::async, [&] { return cvh::copy_settled_rects(&r, 1, st); });
  if (copy.wait_for(std::chrono::seconds(10)) != std::future_status::ready) _exit(1);
  CHECK(copy.get() == CV_OK && host == dev);
  gate.unlock();
}

// Small pieces of caller memory that follow each other in an array on the device
// (those of many meshes) share transfers, in both directions, whatever their
// sizes; what only happens to lie behind the piece before does not.
void check_many() {
  for (bool up : {true, false}) {
    std::vector<std::vector<char>> host;
    std::vector<CallerRect> rects;
    size_t total = 0;
    for (size_t k = 0; k < 20000; k++) {
      // (20000 parts of two arrays of half as many, the first of each empty)
      host.emplace_back(k % 10000 == 0 ? 0 : k == 777 ? 2 * P + 100 : 36 * (1 + k % 50));
      for (size_t j = 0; j < host[k].size(); j++) host[k][j] = (char)(3 * k + j);
      total += host[k].size();
    }
    std::vector<char> dev(total, 'd'), want;
    for (size_t j = 0; !up && j < total; j++) dev[j] = (char)(j * 11 + (j >> 9));
    size_t at = 0, transfers = 0, array = 0;
    for (auto& h : host) {
      rects.push_back(CallerRect::flat(h.data(), dev.data() + at, h.size(), rects.size() % 10000));
      at += h.size();
      array += h.size();
      if (rects.size() % 10000 == 0) {
        transfers += (array + P - 1) / P;
        array = 0;
      }
    }
    fake::transfers = 0;
    CHECK(cvh::copy_caller_rects(rects.data(), rects.size(), up, new_stream()) == CV_OK);
    for (auto& h : host) want.insert(want.end(), h.begin(), h.end());
    CHECK(want == dev);
    CHECK(fake::transfers == transfers);
  }
}

int main(int argc, char** argv) {
  const std::string name = argc > 1 ? argv[1] : "";
  if (name == "shapes")
    check_shapes();
  else if (name == "coherent")
    check_coherent();
  else if (name == "devices")
    check_devices();
  else if (name == "threads")
    check_threads();
  else if (name == "crowd")
    check_crowd();
  else if (name == "settled")
    check_settled();
  else if (name == "many")
    check_many();
  else
    return 2;
  printf("ok\n");
  return 0;
}
