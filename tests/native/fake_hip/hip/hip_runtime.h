// Host stand-in for the few HIP calls of pyro_amd/csrc/hostcopy.hip: copies
// happen at once, an event can only be recorded on a stream of its device.
#pragma once
#include <atomic>
#include <cstdlib>
#include <cstring>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorInvalidHandle = 400 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
using hipDevice_t = int;
struct FakeStream { int dev; };
struct FakeEvent { int dev; };
using hipStream_t = FakeStream *;
using hipEvent_t = FakeEvent *;
constexpr unsigned hipEventDisableTiming = 2, hipHostMallocPortable = 1;

namespace fake {
inline thread_local int current = 0;
inline std::atomic<int> copies{0}, fail_at{-1}, live{0};  // copies made, the one to fail, events and host blocks
}  // namespace fake

inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int *d) { return *d = fake::current, hipSuccess; }
inline hipError_t hipSetDevice(int d) { return fake::current = d, hipSuccess; }
inline hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t *d) { return *d = s->dev, hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  fake::live++;
  return (*p = std::malloc(n)) ? hipSuccess : hipErrorInvalidValue;
}
inline hipError_t hipHostFree(void *p) { return fake::live--, std::free(p), hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  fake::live++;
  return *e = new FakeEvent{fake::current}, hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { return fake::live--, delete e, hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  return e->dev == s->dev ? hipSuccess : hipErrorInvalidHandle;
}
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  if (fake::copies++ == fake::fail_at) return hipErrorInvalidValue;
  return std::memcpy(d, s, n), hipSuccess;
}
