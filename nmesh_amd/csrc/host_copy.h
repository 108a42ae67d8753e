// host_copy.h -- large copies between a caller's (pageable) memory and the
// device through pinned slots of its own, filled and emptied by several threads.
#pragma once
#include <hip/hip_runtime.h>

#include <stddef.h>

namespace nmx {

// The runtime's copy of pageable memory brings 671 MB to the device in 23.5 ms
// and into an array that has no pages yet in 71 (one thread takes the page
// faults), where the link needs 12.  kThreads threads take chunks of the array
// in turn, each with two slots, one filled or emptied while the other is on its
// way: 17.4 and 17.5 ms.  Not for use from two threads at once.
class HostCopy {
 public:
  ~HostCopy() { release(); }
  // device <- host, or host <- device, in order with the stream s; returns when
  // h has been read or written
  hipError_t copy(int device, double *d, const double *h, size_t n, hipStream_t s) {
    return run(device, (char *)d, (char *)h, 8 * n, true, s);
  }
  hipError_t copy_back(int device, double *h, const double *d, size_t n, hipStream_t s) {
    return run(device, (char *)d, (char *)h, 8 * n, false, s);
  }
  void release();

 private:
  static constexpr int kThreads = 8;
  // The plain copy below kMinUp and kMinDown (10.5 MB up 0.35 ms and 0.55 by
  // threads, down 0.81 and 0.60; 35 MB up 1.19 and 1.21, 56 MB 2.0 and 1.65;
  // 4.4 MB down 0.35 and 0.42), and for memory that HIP knows (pinned, managed
  // or the device's).
  static constexpr size_t kMinUp = 40 << 20, kMinDown = 8 << 20, kMaxSlot = 2 << 20;
  hipError_t run(int device, char *d, char *h, size_t bytes, bool up, hipStream_t s);
  hipError_t setup(size_t bytes);
  char *pin = nullptr;          // the slots
  size_t pinned = 0;
  hipEvent_t ev[2 * kThreads] = {};
};

}  // namespace nmx
