// Drives HostCopy (nmesh_amd/csrc/host_copy.cpp) on the CPU against stand-ins
// for the HIP calls it makes: "device" memory is host memory, copies are done
// when they are queued.  argv[1]: threads (allocations beyond the first few
// throwing std::bad_alloc, as a machine out of memory does), memcpy (a queued
// copy fails) or round (copies both ways of sizes around the slots').
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "../nmesh_amd/csrc/host_copy.h"

static std::atomic<long> allocs_left{-1};   // -1: unlimited
static std::atomic<int> copies{0};
static int fail_copy = -1;

void *operator new(size_t n) {
  if (allocs_left >= 0 && allocs_left-- <= 0) {
    allocs_left = 0;
    throw std::bad_alloc();
  }
  if (void *p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" {
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return (*p = std::malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)std::malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { std::free((void *)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return hipErrorInvalidValue; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  if (copies++ == fail_copy) return hipErrorUnknown;
  std::memcpy(d, s, n);
  return hipSuccess;
}
}

static int round_trip(size_t n, bool limited) {
  std::vector<double> h(n), d(n), back(n);
  for (size_t i = 0; i < n; ++i) h[i] = (double)i + 0.5;
  nmx::HostCopy io;
  if (limited) allocs_left = 3;
  hipError_t e = io.copy(0, d.data(), h.data(), n, nullptr);
  if (limited) allocs_left = 3;
  if (e == hipSuccess) e = io.copy_back(0, back.data(), d.data(), n, nullptr);
  allocs_left = -1;
  if (e != hipSuccess) return std::printf("error %d\n", (int)e), 1;
  if (std::memcmp(h.data(), d.data(), 8 * n) || std::memcmp(h.data(), back.data(), 8 * n))
    return std::printf("%zu values: wrong\n", n), 1;
  return 0;
}

int main(int, char **argv) {
  const std::string what = argv[1];
  const size_t up = (40 << 20) / 8, down = (8 << 20) / 8, slot = (2 << 20) / 8;
  if (what == "threads") return round_trip(up + 1, true);
  if (what == "memcpy") {
    std::vector<double> h(up + 1), d(up + 1);
    nmx::HostCopy io;
    for (fail_copy = 0; fail_copy < 21; ++fail_copy) {
      copies = 0;
      if (io.copy(0, d.data(), h.data(), h.size(), nullptr) != hipErrorUnknown)
        return std::printf("copy %d failed without an error\n", fail_copy), 1;
    }
    return 0;
  }
  for (size_t n : {(size_t)1, down - 1, down, down + 1, up - 1, up, up + 1, up + slot, up + slot + 3})
    if (round_trip(n, false)) return 1;
  return 0;
}
