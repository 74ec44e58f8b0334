// ads_staging.hip -- see ads_staging.h. Host code only.
#include "ads_staging.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>
#include <vector>

namespace f3d {
namespace host {
namespace {

// memcpy by several threads, which live as long as one transfer: they wait
// for pieces by polling, so that a piece costs no thread start and no system
// call. Without helpers (none wanted, or none to be had) copy() is memcpy.
class ParallelCopy {
 public:
  explicit ParallelCopy(size_t bytes) {
    // a helper per 4 MB of the transfer, at most 7, and half of the CPUs
    const unsigned hw = std::max(2u, std::thread::hardware_concurrency());
    const size_t want = std::min<size_t>({bytes >> 22, 7, hw / 2 - 1});
    try {
      helpers_.reserve(want);
      for (size_t h = 0; h < want; ++h) helpers_.emplace_back([this, h] { work(h + 1); });
    } catch (const std::exception &) {  // fewer threads than wanted
    }
    parts_ = helpers_.size() + 1;
    open_.store(true, std::memory_order_release);
  }
  ~ParallelCopy() {
    piece_.store(-1, std::memory_order_release);
    for (auto &t : helpers_) t.join();
  }
  ParallelCopy(const ParallelCopy &) = delete;
  ParallelCopy &operator=(const ParallelCopy &) = delete;

  void copy(void *dst, const void *src, size_t n) {
    dst_ = (char *)dst;
    src_ = (const char *)src;
    n_ = n;
    left_.store(helpers_.size(), std::memory_order_relaxed);
    piece_.fetch_add(1, std::memory_order_release);
    part(0);
    while (left_.load(std::memory_order_acquire) != 0) std::this_thread::yield();
  }

 private:
  void part(size_t h) {
    const size_t step = (n_ / parts_ + 63) & ~(size_t)63;  // whole cache lines
    const size_t a = std::min(n_, h * step), b = h + 1 == parts_ ? n_ : std::min(n_, (h + 1) * step);
    if (b > a) memcpy(dst_ + a, src_ + a, b - a);
  }
  void work(size_t h) {
    while (!open_.load(std::memory_order_acquire)) std::this_thread::yield();
    long seen = 0;
    for (;;) {
      const long p = piece_.load(std::memory_order_acquire);
      if (p < 0) return;
      if (p == seen) {
        std::this_thread::yield();
        continue;
      }
      seen = p;
      part(h);
      left_.fetch_sub(1, std::memory_order_release);
    }
  }

  std::vector<std::thread> helpers_;
  size_t parts_ = 1, n_ = 0;
  char *dst_ = nullptr;
  const char *src_ = nullptr;
  std::atomic<bool> open_{false};  // parts_ is final
  std::atomic<long> piece_{0};     // pieces handed out; -1: no more
  std::atomic<size_t> left_{0};    // helpers still copying
};

// Whether the runtime takes the transfer as it is: host memory that it can
// reach directly, or a stream under capture, where nothing may be waited for.
bool direct(const void *p, hipStream_t st) {
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) return true;
  hipPointerAttribute_t a;
  memset(&a, 0, sizeof(a));
  const bool known = hipPointerGetAttributes(&a, p) == hipSuccess && a.type != hipMemoryTypeUnregistered;
  (void)hipGetLastError();  // an address the runtime does not know is no error here
  return known;
}

}  // namespace

void Staging::release() {
  for (int q = 0; q < kBuffers; ++q) {
    if (done[q]) (void)hipEventSynchronize(done[q]), (void)hipEventDestroy(done[q]);
    if (buf[q]) (void)hipHostFree(buf[q]);
    done[q] = nullptr;
    buf[q] = nullptr;
  }
}

bool Staging::ready() {
  if (done[kBuffers - 1]) return true;
  for (int q = 0; q < kBuffers; ++q)
    if (hipHostMalloc(&buf[q], kPiece, hipHostMallocDefault) != hipSuccess ||
        hipEventCreateWithFlags(&done[q], hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      release();
      return false;
    }
  return true;
}

hipError_t Staging::in(void *dst, const void *src, size_t bytes, hipStream_t st) {
  if (bytes < kLeast || direct(src, st) || !ready()) return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st);
  ParallelCopy par(bytes);
  int q = 0;
  for (size_t at = 0; at < bytes; at += kPiece, q = (q + 1) % kBuffers) {
    const size_t n = std::min(kPiece, bytes - at);
    hipError_t e = hipEventSynchronize(done[q]);  // the buffer's last transfer (none yet: returns at once)
    if (e != hipSuccess) return e;
    par.copy(buf[q], (const char *)src + at, n);
    e = hipMemcpyAsync((char *)dst + at, buf[q], n, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hipEventRecord(done[q], st);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t Staging::out(void *dst, const void *src, size_t bytes, hipStream_t st) {
  if (bytes < kLeast || direct(dst, st) || !ready()) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
    return e == hipSuccess ? hipStreamSynchronize(st) : e;
  }
  ParallelCopy par(bytes);
  const size_t pieces = (bytes + kPiece - 1) / kPiece;
  auto length = [&](size_t p) { return std::min(kPiece, bytes - p * kPiece); };
  // kBuffers - 1 transfers ahead of the piece that is copied out
  for (size_t p = 0; p < pieces + kBuffers - 1; ++p) {
    if (p < pieces) {
      const int q = (int)(p % kBuffers);
      hipError_t e = hipEventSynchronize(done[q]);  // an earlier call's transfer out of the buffer
      if (e == hipSuccess) e = hipMemcpyAsync(buf[q], (const char *)src + p * kPiece, length(p), hipMemcpyDeviceToHost, st);
      if (e == hipSuccess) e = hipEventRecord(done[q], st);
      if (e != hipSuccess) return e;
    }
    if (p + 1 >= kBuffers) {
      const size_t r = p + 1 - kBuffers;
      const hipError_t e = hipEventSynchronize(done[r % kBuffers]);
      if (e != hipSuccess) return e;
      par.copy((char *)dst + r * kPiece, buf[r % kBuffers], length(r));
    }
  }
  return hipSuccess;
}

}  // namespace host
}  // namespace f3d
