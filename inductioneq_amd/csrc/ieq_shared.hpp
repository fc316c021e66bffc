// Ordering of the buffers that belong to a program (not to a call's arguments) between the streams it is used on.
#pragma once

#include <hip/hip_runtime.h>

namespace ieq {

// Calls on one stream follow one another; when the program is given another stream, the end of what has used its
// buffers is marked on the old one, and the next call that uses them waits for it.  (A mark after every call costs
// 3 to 5 us of a call: 32^3 FP32, one 2N step, 76 -> 82 us.)  A stream that records a graph can neither mark
// nor wait; its replays are the caller's to order.
struct SharedUse {
  hipEvent_t done = nullptr;
  bool used = false;  // on the program's present stream
  bool wait = false;  // `done` is still to be waited for

  static bool capturing(hipStream_t s) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) == hipSuccess) return cap != hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return true;
  }
  // The program leaves stream `old`.
  void leave(hipStream_t old) {
    if (!used || capturing(old)) return;
    if (!done && hipEventCreateWithFlags(&done, hipEventDisableTiming) != hipSuccess) done = nullptr;
    if (done && hipEventRecord(done, old) == hipSuccess) {
      wait = true;
    } else {
      (void)hipStreamSynchronize(old);
      (void)hipGetLastError();
    }
    used = false;
  }
  // A call on `s`, which records no graph, is about to use a buffer.
  bool enter(hipStream_t s) {
    if (wait && hipStreamWaitEvent(s, done, 0) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    wait = false;
    return used = true;
  }
  ~SharedUse() {
    if (done) (void)hipEventDestroy(done);
  }
};

}  // namespace ieq
