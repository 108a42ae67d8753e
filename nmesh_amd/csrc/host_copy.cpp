// host_copy.cpp -- copies through pinned slots (host_copy.h).
#include "host_copy.h"

#include <string.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <thread>

namespace nmx {

void HostCopy::release() {
  if (pin) (void)hipHostFree(pin);
  pin = nullptr;
  for (auto &e : ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  pinned = 0;
}

hipError_t HostCopy::setup(size_t bytes) {
  if (bytes <= pinned) return hipSuccess;
  release();
  hipError_t e = hipHostMalloc((void **)&pin, bytes, hipHostMallocDefault);
  for (auto &v : ev)
    if (e == hipSuccess) e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
  if (e != hipSuccess) release();
  else pinned = bytes;
  return e;
}

hipError_t HostCopy::run(int device, char *d, char *h, size_t bytes, bool up, hipStream_t s) {
  const size_t slot_bytes = std::min(kMaxSlot, (bytes / 16 + 4096) / 4096 * 4096);
  const size_t chunks = (bytes + slot_bytes - 1) / slot_bytes;
  const int nt = (int)std::min<size_t>(chunks, kThreads);
  bool plain = bytes < (up ? kMinUp : kMinDown);
  if (!plain) {
    hipPointerAttribute_t at;
    plain = hipPointerGetAttributes(&at, h) == hipSuccess && at.type != hipMemoryTypeUnregistered;
    if (!plain) plain = setup(2 * nt * slot_bytes) != hipSuccess;
    (void)hipGetLastError();   // of memory that HIP does not know, or none to pin
  }
  if (plain) {
    hipError_t e = hipMemcpyAsync(up ? d : h, up ? h : d, bytes, up ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, s);
    return e == hipSuccess ? hipStreamSynchronize(s) : e;
  }
  std::atomic<size_t> next{0};
  std::atomic<int> err{hipSuccess};
  auto work = [&](int t) {
    hipError_t e = hipSetDevice(device);
    char *slot[2] = {pin + 2 * t * slot_bytes, pin + (2 * t + 1) * slot_bytes};
    size_t held[2] = {(size_t)-1, (size_t)-1};   // chunk on its way in each slot
    auto len = [&](size_t c) { return std::min(slot_bytes, bytes - c * slot_bytes); };
    auto settle = [&](int k) {
      if (held[k] == (size_t)-1) return;
      const hipError_t w = hipEventSynchronize(ev[2 * t + k]);
      if (e == hipSuccess) e = w;
      if (!up && e == hipSuccess) memcpy(h + held[k] * slot_bytes, slot[k], len(held[k]));
      held[k] = (size_t)-1;
    };
    int k = 0;
    for (;; k ^= 1) {
      settle(k);
      const size_t c = e == hipSuccess && err == hipSuccess ? next++ : chunks;
      if (c >= chunks) break;
      if (up) memcpy(slot[k], h + c * slot_bytes, len(c));
      e = hipMemcpyAsync(up ? d + c * slot_bytes : slot[k], up ? slot[k] : d + c * slot_bytes, len(c),
                         up ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, s);
      if (e == hipSuccess) e = hipEventRecord(ev[2 * t + k], s);
      if (e == hipSuccess) held[k] = c;
      else (void)hipStreamSynchronize(s);   // nothing of this thread in flight
    }
    settle(k ^ 1);
    if (e != hipSuccess) err = e;
  };
  std::thread th[kThreads];
  int started = 1;
  try {
    for (; started < nt; ++started) th[started] = std::thread(work, started);
  } catch (const std::exception &) {
    // no thread, or no memory for its start: fewer threads take all chunks
  }
  work(0);
  for (int t = 1; t < started; ++t) th[t].join();
  return (hipError_t)err.load();
}

}  // namespace nmx
