// host_pipe.cpp -- read-back through pinned buffers.
//
// hipMemcpyAsync into pageable memory runs at 16 GB/s here, into pinned
// memory at 55 GB/s; the caller's array (a fresh numpy array, a C++ vector)
// is pageable and may not be registered, so the bytes go through two pinned
// chunks per worker, the copy of one overlapping the host copy of the other.
// Large reads are bound by the host copy (first touches of the caller's
// pages included), so up to kWorkers threads take contiguous parts.
#include "host_pipe.hpp"

#include <algorithm>
#include <cstring>
#include <exception>
#include <map>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "domain.hpp"

namespace wake_hip {

namespace {

constexpr size_t kChunk = 1u << 20;
constexpr size_t kPerWorker = 4u << 20;  // a worker's part at least
constexpr size_t kWorkers = 4;
constexpr size_t kKept = 8;  // idle buffers kept per device

struct Stage {
  char* p[2] = {nullptr, nullptr};
  hipEvent_t e[2] = {nullptr, nullptr};
  Stage() {
    try {
      for (int k = 0; k < 2; ++k) {
        check(hipHostMalloc(reinterpret_cast<void**>(&p[k]), kChunk, hipHostMallocDefault), "hipHostMalloc");
        check(hipEventCreateWithFlags(&e[k], hipEventDisableTiming), "event");
      }
    } catch (...) {
      drop();
      throw;
    }
  }
  ~Stage() { drop(); }
  Stage(const Stage&) = delete;
  Stage& operator=(const Stage&) = delete;

 private:
  void drop() {
    for (int k = 0; k < 2; ++k) {
      if (p[k]) (void)hipHostFree(p[k]);
      if (e[k]) (void)hipEventDestroy(e[k]);
      p[k] = nullptr;
      e[k] = nullptr;
    }
    (void)hipGetLastError();
  }
};

// Idle buffers by device; never destroyed with the process (the runtime may
// be gone by then).
struct Pool {
  std::mutex m;
  std::map<int, std::vector<std::unique_ptr<Stage>>> idle;
};
Pool& pool() {
  static Pool* p = new Pool;
  return *p;
}

std::unique_ptr<Stage> take(int dev) {
  {
    std::lock_guard<std::mutex> lk(pool().m);
    auto& v = pool().idle[dev];
    if (!v.empty()) {
      std::unique_ptr<Stage> s = std::move(v.back());
      v.pop_back();
      return s;
    }
  }
  return std::make_unique<Stage>();
}

void give(int dev, std::unique_ptr<Stage> s) {
  std::lock_guard<std::mutex> lk(pool().m);
  auto& v = pool().idle[dev];
  if (v.size() < kKept) v.push_back(std::move(s));
}

void copy_part(char* dst, const char* src, size_t bytes, hipStream_t stream, int dev) {
  std::unique_ptr<Stage> s = take(dev);
  try {
    const size_t n = (bytes + kChunk - 1) / kChunk;
    auto issue = [&](size_t i) {
      const size_t at = i * kChunk, len = std::min(kChunk, bytes - at);
      check(hipMemcpyAsync(s->p[i & 1], src + at, len, hipMemcpyDeviceToHost, stream), "d2h");
      check(hipEventRecord(s->e[i & 1], stream), "event");
    };
    if (n > 0) issue(0);
    for (size_t i = 0; i < n; ++i) {
      if (i + 1 < n) issue(i + 1);
      check(hipEventSynchronize(s->e[i & 1]), "d2h");
      const size_t at = i * kChunk;
      std::memcpy(dst + at, s->p[i & 1], std::min(kChunk, bytes - at));
    }
  } catch (...) {
    (void)hipStreamSynchronize(stream);  // nothing may still write the buffers
    throw;
  }
  give(dev, std::move(s));
}

}  // namespace

void device_to_host(void* dst, const void* src, size_t bytes, hipStream_t stream) {
  int dev = 0;
  check(hipGetDevice(&dev), "hipGetDevice");
  const size_t workers = std::max<size_t>(1, std::min(kWorkers, bytes / kPerWorker));
  char* d = static_cast<char*>(dst);
  const char* p = static_cast<const char*>(src);
  const size_t part = (bytes / workers + 4095) / 4096 * 4096;
  std::vector<std::exception_ptr> errors(workers);
  std::vector<std::thread> threads;
  auto work = [&](size_t w) {
    try {
      const size_t at = std::min(bytes, w * part), end = w + 1 == workers ? bytes : std::min(bytes, at + part);
      if (w > 0) check(hipSetDevice(dev), "hipSetDevice");
      copy_part(d + at, p + at, end - at, stream, dev);
    } catch (...) {
      errors[w] = std::current_exception();
    }
  };
  size_t started = 1;
  try {
    for (; started < workers; ++started) threads.emplace_back(work, started);
  } catch (...) {
    // no thread to be had: the parts left are taken here
  }
  work(0);
  for (size_t w = started; w < workers; ++w) work(w);
  for (std::thread& t : threads) t.join();
  for (const std::exception_ptr& e : errors)
    if (e) std::rethrow_exception(e);
}

void trim_host_pipe() noexcept {
  std::lock_guard<std::mutex> lk(pool().m);
  pool().idle.clear();
}

}  // namespace wake_hip
