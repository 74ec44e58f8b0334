// ads_staging.h -- copies between host arrays and the device (internal).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace f3d {
namespace host {

// Transfers of large pageable arrays through page-locked buffers. A context
// holds one object while it lives; the buffers are shared by all contexts.
//
// The runtime moves a pageable array through small buffers of its own with
// one copying thread, which bounds the transfer. Here the array moves through
// kBuffers buffers of kPiece bytes: a few threads copy a piece to or from one
// buffer while the others are in transfer. An x, a y and a z sweep on host
// arrays at 200 x 150 x 50 x 8, FP32 (0.37 GB between host and device): 18.8 ->
// 10.8 ms; the output products of 360 x 240 x 60 x 10: 19 to 27 -> 5.2.
//
// A transfer takes a set of buffers for its length, from any thread; at most
// kIdle sets of a device wait for the next one (96 MiB, however many contexts
// there are), and the last context to go gives them back.
class Staging {
 public:
  static constexpr int kBuffers = 3;
  static constexpr size_t kPiece = (size_t)8 << 20;
  static constexpr size_t kIdle = 4;
  // arrays below this size go to the runtime as they are
  static constexpr size_t kLeast = (size_t)2 << 20;

  Staging();
  ~Staging();
  Staging(const Staging &) = delete;
  Staging &operator=(const Staging &) = delete;

  // dst (device) = src (host). On return src may be changed or freed unless it
  // is page-locked; the transfer is ordered on the stream.
  hipError_t in(void *dst, const void *src, size_t bytes, hipStream_t st);
  // dst (host) = src (device), complete on return; with wait false at the
  // latest when the stream has been waited for (small arrays then share a wait)
  hipError_t out(void *dst, const void *src, size_t bytes, hipStream_t st, bool wait = true);
};

}  // namespace host
}  // namespace f3d
