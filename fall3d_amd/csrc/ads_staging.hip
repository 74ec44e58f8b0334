// ads_staging.hip -- see ads_staging.h. Host code only.
#include "ads_staging.h"

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace f3d {
namespace host {
namespace {

// memcpy by several threads, which live as long as one transfer. They wait for
// a piece by polling for kPoll, the time between pieces while the bus is busy,
// and sleep beyond it: a transfer may wait behind other work of its stream
// (a read-back behind 1200 steps of 360 x 240 x 60 x 10, 0.54 s: 4.2 s of CPU time
// when they polled all the while, 0.65 s now, most of it the runtime's own wait).
// Without helpers (none wanted, or none to be had) copy() is memcpy.
class ParallelCopy {
 public:
  explicit ParallelCopy(size_t bytes) {
    // a helper per 4 MB of the transfer, at most 7, and half of the process's CPUs
    const unsigned hw = std::max(2u, std::thread::hardware_concurrency());
    const size_t want = std::min<size_t>({bytes >> 22, 7, hw / 2 - 1});
    try {
      helpers_.reserve(want);
      for (size_t h = 0; h < want; ++h) helpers_.emplace_back([this, h] { work(h + 1); });
    } catch (const std::exception &) {  // fewer threads than wanted
    }
  }
  ~ParallelCopy() {
    hand_out(-1);
    for (auto &t : helpers_) t.join();
  }
  ParallelCopy(const ParallelCopy &) = delete;
  ParallelCopy &operator=(const ParallelCopy &) = delete;

  void copy(void *dst, const void *src, size_t n) {
    dst_ = (char *)dst;
    src_ = (const char *)src;
    n_ = n;
    left_.store(helpers_.size(), std::memory_order_relaxed);
    hand_out(++pieces_);
    part(0);
    while (left_.load(std::memory_order_acquire) != 0) std::this_thread::yield();
  }

 private:
  static constexpr std::chrono::microseconds kPoll{200};

  void hand_out(long p) {
    {
      std::lock_guard<std::mutex> lk(mu_);
      piece_.store(p, std::memory_order_release);
    }
    wake_.notify_all();
  }
  void part(size_t h) {
    const size_t parts = helpers_.size() + 1, step = (n_ / parts + 63) & ~(size_t)63;  // whole cache lines
    const size_t a = std::min(n_, h * step), b = h + 1 == parts ? n_ : std::min(n_, (h + 1) * step);
    if (b > a) memcpy(dst_ + a, src_ + a, b - a);
  }
  // the piece after `seen`, -1: no more
  long next(long seen) {
    const auto until = std::chrono::steady_clock::now() + kPoll;
    do {
      const long p = piece_.load(std::memory_order_acquire);
      if (p != seen) return p;
      std::this_thread::yield();
    } while (std::chrono::steady_clock::now() < until);
    std::unique_lock<std::mutex> lk(mu_);
    wake_.wait(lk, [&] { return piece_.load(std::memory_order_acquire) != seen; });
    return piece_.load(std::memory_order_acquire);
  }
  void work(size_t h) {
    for (long seen = 0; (seen = next(seen)) >= 0;) {
      part(h);  // (helpers_ is complete: the first piece comes after the constructor)
      left_.fetch_sub(1, std::memory_order_release);
    }
  }

  std::vector<std::thread> helpers_;
  std::mutex mu_;
  std::condition_variable wake_;
  size_t n_ = 0;
  char *dst_ = nullptr;
  const char *src_ = nullptr;
  long pieces_ = 0;
  std::atomic<long> piece_{0};     // pieces handed out; -1: no more
  std::atomic<size_t> left_{0};    // helpers still copying
};

// Page-locked buffers of one transfer at a time, for one device.
struct Buffers {
  int device;
  void *buf[Staging::kBuffers] = {};
  hipEvent_t done[Staging::kBuffers] = {};  // the buffer's last transfer
  bool used = false;                        // the events have been recorded
  hipStream_t stream = nullptr;             // the last transfer's (compared, never used)
  explicit Buffers(int dev) : device(dev) {}
  ~Buffers() {
    for (int q = 0; q < Staging::kBuffers; ++q) {
      if (done[q]) (void)hipEventSynchronize(done[q]), (void)hipEventDestroy(done[q]);
      if (buf[q]) (void)hipHostFree(buf[q]);
    }
  }
  bool allocate() {
    for (int q = 0; q < Staging::kBuffers; ++q)
      if (hipHostMalloc(&buf[q], Staging::kPiece, hipHostMallocDefault) != hipSuccess ||
          hipEventCreateWithFlags(&done[q], hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
    return true;
  }
  bool over() const {  // no transfer of an earlier call is under way
    if (!used) return true;
    for (hipEvent_t e : done)
      if (hipEventQuery(e) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
    return true;
  }
};
using Set = std::unique_ptr<Buffers>;

// The sets that wait for a transfer, kIdle of a device at most.
class Pool {
 public:
  // A set of the current device for a transfer on st: one whose transfers are
  // over or on the same stream (two contexts' streams do not wait for each
  // other), else a new one while fewer than kIdle wait, else any. Null: none to
  // be had.
  Set take(hipStream_t st) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kDevices) return nullptr;
    {
      std::lock_guard<std::mutex> lk(mu_);
      size_t waiting = 0;
      for (Set &s : idle_[dev]) {
        if (s && (s->stream == st || s->over())) return std::move(s);
        waiting += s ? 1 : 0;
      }
      if (waiting == Staging::kIdle) return std::move(idle_[dev][0]);
    }
    Set s(new (std::nothrow) Buffers(dev));
    if (!s || !s->allocate()) return nullptr;
    return s;
  }
  void give(Set s, hipStream_t st) {
    s->used = true;
    s->stream = st;
    std::lock_guard<std::mutex> lk(mu_);
    if (users_ == 0) return;
    for (Set &slot : idle_[s->device])
      if (!slot) {
        slot = std::move(s);
        return;
      }
  }  // (a set without a place goes with s)
  void join() {
    std::lock_guard<std::mutex> lk(mu_);
    ++users_;
  }
  void leave() {
    std::array<std::array<Set, Staging::kIdle>, kDevices> last;
    std::lock_guard<std::mutex> lk(mu_);
    if (--users_ == 0) last.swap(idle_);
  }

 private:
  static constexpr int kDevices = 64;
  std::mutex mu_;
  std::array<std::array<Set, Staging::kIdle>, kDevices> idle_;
  long users_ = 0;
};
// never destroyed: a context that outlives main keeps its buffers until the process ends
Pool &pool() {
  static Pool &p = *new Pool;
  return p;
}

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

Staging::Staging() { pool().join(); }
Staging::~Staging() { pool().leave(); }

hipError_t Staging::in(void *dst, const void *src, size_t bytes, hipStream_t st) {
  Set s = bytes < kLeast || direct(src, st) ? nullptr : pool().take(st);
  if (!s) return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st);
  hipError_t e = hipSuccess;
  {
    ParallelCopy par(bytes);
    int q = 0;
    for (size_t at = 0; at < bytes && e == hipSuccess; at += kPiece, q = (q + 1) % kBuffers) {
      const size_t n = std::min(kPiece, bytes - at);
      e = hipEventSynchronize(s->done[q]);  // the buffer's last transfer (none yet: returns at once)
      if (e != hipSuccess) break;
      par.copy(s->buf[q], (const char *)src + at, n);
      e = hipMemcpyAsync((char *)dst + at, s->buf[q], n, hipMemcpyHostToDevice, st);
      if (e == hipSuccess) e = hipEventRecord(s->done[q], st);
    }
  }
  pool().give(std::move(s), st);
  return e;
}

hipError_t Staging::out(void *dst, const void *src, size_t bytes, hipStream_t st, bool wait) {
  Set s = bytes < kLeast || direct(dst, st) ? nullptr : pool().take(st);
  if (!s) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
    return e == hipSuccess && wait ? hipStreamSynchronize(st) : e;
  }
  hipError_t e = hipSuccess;
  {
    ParallelCopy par(bytes);  // its threads start while the first transfer runs
    const size_t pieces = (bytes + kPiece - 1) / kPiece;
    auto length = [&](size_t p) { return std::min(kPiece, bytes - p * kPiece); };
    // kBuffers - 1 transfers ahead of the piece that is copied out
    for (size_t p = 0; p < pieces + kBuffers - 1 && e == hipSuccess; ++p) {
      if (p < pieces) {
        const int q = (int)(p % kBuffers);
        e = hipEventSynchronize(s->done[q]);  // an earlier call's transfer through the buffer
        if (e == hipSuccess) e = hipMemcpyAsync(s->buf[q], (const char *)src + p * kPiece, length(p), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipEventRecord(s->done[q], st);
      }
      if (p + 1 >= kBuffers && e == hipSuccess) {
        const size_t r = p + 1 - kBuffers;
        e = hipEventSynchronize(s->done[r % kBuffers]);
        if (e != hipSuccess) break;
        par.copy((char *)dst + r * kPiece, s->buf[r % kBuffers], length(r));
      }
    }
  }
  pool().give(std::move(s), st);
  return e;
}

}  // namespace host
}  // namespace f3d
