// scratch.h — device scratch of the kernel-layer entry points that need some beside
// their caller's buffers (row products: prepared activations and K-split partials;
// decode attention: split partials).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

namespace uaii {

// One call's hold on a scratch buffer of the current device, for launches on `stream`.
// Construct it, reserve(), enqueue everything that touches data() on `stream`, and let
// it go out of scope; nothing waits for the launches. Buffers are kept for later calls:
//   null stream       one buffer. Its work runs in order, so nothing else is needed.
//   other streams     up to kSlots buffers. Each carries an event recorded after its
//                     last call, which a call on another stream waits for on the device.
//   streams in capture  a buffer that only captured calls use and that is never freed:
//                     a graph holds its address for as long as the graph lives. All
//                     captured calls share it, so a program orders replays (and branches
//                     of one capture) that hold such calls.
// Buffers grow to the largest request. Where the device has no memory left for one, the
// idle slots are freed first.
class Scratch {
 public:
  static constexpr int kSlots = 4;

  explicit Scratch(hipStream_t stream);
  ~Scratch();
  Scratch(const Scratch&) = delete;
  Scratch& operator=(const Scratch&) = delete;

  // data() of at least `bytes` (at a 256-byte boundary). After a failure a smaller
  // request may be tried.
  hipError_t reserve(size_t bytes);
  char* data() const { return data_; }
  // The stream is being captured into a graph.
  bool capturing() const { return capturing_; }

  struct Slot;

 private:
  std::unique_lock<std::mutex> lock_;  // held until the call's launches are enqueued
  hipStream_t stream_;
  bool capturing_ = false;
  Slot* slot_ = nullptr;  // of a stream other than the null stream, to be marked busy
  char* data_ = nullptr;
};

}  // namespace uaii
