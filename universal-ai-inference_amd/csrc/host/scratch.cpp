#include "scratch.h"

#include <algorithm>
#include <cstdint>

namespace uaii {

struct Scratch::Slot {
  void* p = nullptr;
  size_t bytes = 0;
  hipEvent_t done = nullptr;   // after the slot's last call; null: never used
  hipStream_t last = nullptr;  // that call's stream, to prefer the slot by; never taken for an order
  uint64_t turn = 0;           // when that call was
};

// The `done` events carry no system-scope fence, which costs every call of a side stream
// (9 rows of 512 x 512: 14.4 us with no event at all, 16.4 with a fence, 15.3 without).
// A slot's change of stream adds one: the event `fence` on the new stream, which writes
// the caches back before that stream's first launch.
namespace {

constexpr int kMaxDevices = 64;

struct Device {
  void* null_p = nullptr;
  size_t null_bytes = 0;
  Scratch::Slot slots[Scratch::kSlots];
  hipEvent_t fence = nullptr;
  void* cap_p = nullptr;
  size_t cap_bytes = 0;
  uint64_t turn = 0;
};

std::mutex g_mu;
Device g_dev[kMaxDevices];

bool null_stream(hipStream_t s) { return s == nullptr || s == hipStreamLegacy; }

bool idle(const Scratch::Slot& s) {
  if (!s.done) return true;
  if (hipEventQuery(s.done) == hipSuccess) return true;
  (void)hipGetLastError();  // not ready
  return false;
}

hipError_t allocate(Device& d, size_t bytes, void** p) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipErrorOutOfMemory) return e;
  (void)hipGetLastError();
  for (Scratch::Slot& s : d.slots) {
    if (!s.p || !idle(s)) continue;
    (void)hipFree(s.p);
    s.p = nullptr;
    s.bytes = 0;
  }
  return hipMalloc(p, bytes);
}

// hipMalloc records nothing, and a thread in relaxed mode may call it during a capture.
hipError_t allocate_in_capture(size_t bytes, void** p) {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  hipError_t e = hipThreadExchangeStreamCaptureMode(&mode);
  if (e != hipSuccess) return e;
  e = hipMalloc(p, bytes);
  (void)hipThreadExchangeStreamCaptureMode(&mode);
  return e;
}

hipError_t new_event(hipEvent_t* ev, unsigned flags) {
  const hipError_t e = hipEventCreateWithFlags(ev, hipEventDisableTiming | flags);
  if (e != hipSuccess) *ev = nullptr;
  return e;
}

// `stream`'s own slot, else an idle one, else the one used longest ago.
Scratch::Slot* pick(Device& d, hipStream_t stream) {
  for (Scratch::Slot& s : d.slots)
    if (s.done && s.last == stream) return &s;
  for (Scratch::Slot& s : d.slots)
    if (idle(s)) return &s;
  return std::min_element(d.slots, d.slots + Scratch::kSlots,
                          [](const Scratch::Slot& a, const Scratch::Slot& b) { return a.turn < b.turn; });
}

}  // namespace

Scratch::Scratch(hipStream_t stream) : lock_(g_mu), stream_(stream) {
  if (null_stream(stream)) return;  // cannot be captured
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  capturing_ = hipStreamIsCapturing(stream, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone;
}

hipError_t Scratch::reserve(size_t bytes) {
  int id = 0;
  hipError_t e = hipGetDevice(&id);
  if (e != hipSuccess) return e;
  if (id < 0 || id >= kMaxDevices) return hipErrorInvalidDevice;
  Device& d = g_dev[id];
  if (capturing_) {
    if (bytes > d.cap_bytes) {
      // at least doubled: all that earlier graphs hold stays below the newest buffer
      const size_t want = std::max(bytes, 2 * d.cap_bytes);
      void* p = nullptr;
      e = allocate_in_capture(want, &p);
      if (e != hipSuccess) return e;
      d.cap_p = p;
      d.cap_bytes = want;
    }
    data_ = static_cast<char*>(d.cap_p);
    return hipSuccess;
  }
  if (null_stream(stream_)) {
    if (bytes > d.null_bytes) {
      if (d.null_p) {
        e = hipStreamSynchronize(stream_);
        if (e != hipSuccess) return e;
        (void)hipFree(d.null_p);
        d.null_p = nullptr;
        d.null_bytes = 0;
      }
      e = allocate(d, bytes, &d.null_p);
      if (e != hipSuccess) return e;
      d.null_bytes = bytes;
    }
    data_ = static_cast<char*>(d.null_p);
    return hipSuccess;
  }
  Slot* s = pick(d, stream_);
  if (!s->done) {
    e = new_event(&s->done, hipEventDisableSystemFence);
    if (e != hipSuccess) return e;
  } else if (bytes > s->bytes && s->p) {
    e = hipEventSynchronize(s->done);
    if (e != hipSuccess) return e;
    (void)hipFree(s->p);
    s->p = nullptr;
    s->bytes = 0;
  } else {
    e = hipStreamWaitEvent(stream_, s->done, 0);
    if (e == hipSuccess && s->last != stream_) {
      if (!d.fence) e = new_event(&d.fence, 0);
      if (e == hipSuccess) e = hipEventRecord(d.fence, stream_);
    }
    if (e != hipSuccess) return e;
  }
  if (!s->p) {
    e = allocate(d, bytes, &s->p);
    if (e != hipSuccess) return e;
    s->bytes = bytes;
  }
  s->last = stream_;
  s->turn = ++d.turn;
  slot_ = s;
  data_ = static_cast<char*>(s->p);
  return hipSuccess;
}

Scratch::~Scratch() {
  if (slot_ && hipEventRecord(slot_->done, stream_) != hipSuccess) {
    // no event to wait for: the next call must find the slot idle
    (void)hipDeviceSynchronize();
    (void)hipGetLastError();
  }
}

}  // namespace uaii
