// A HIP runtime on host memory for tests of the engine's host code: every call
// completes at once, "device" memory is malloc'd, and the test decides what runs
// out.  Kernel launchers are defined by the tests that reach them; any other
// stays unresolved and ends the test with a segmentation fault.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>

namespace fake {
inline std::map<void*, size_t> dev, pinned;  // live allocations
inline size_t dev_limit = ~size_t(0), dev_used = 0;
inline long n_malloc = 0, n_free = 0, n_sync = 0;
inline hipError_t last = hipSuccess;
inline std::set<hipStream_t> streams, capturing;
inline hipError_t fail(hipError_t e) {
  last = e;
  return e;
}
}  // namespace fake

#define CHECK(c)                                                   \
  do {                                                             \
    if (!(c)) {                                                    \
      std::printf("%s:%d: %s does not hold\n", __FILE__, __LINE__, #c); \
      std::exit(1);                                                \
    }                                                              \
  } while (0)

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  ++fake::n_malloc;
  if (fake::dev_used + n > fake::dev_limit) return fake::fail(hipErrorOutOfMemory);
  *p = std::malloc(n ? n : 1);
  fake::dev[*p] = n;
  fake::dev_used += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  CHECK(fake::dev.count(p));
  ++fake::n_free;
  fake::dev_used -= fake::dev[p];
  fake::dev.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned int) {
  *p = std::malloc(n ? n : 1);
  fake::pinned[*p] = n;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  CHECK(fake::pinned.count(p));
  fake::pinned.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memmove(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { std::memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned int) {
  *s = (hipStream_t)std::malloc(1);
  fake::streams.insert(*s);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  CHECK(fake::streams.count(s));
  fake::streams.erase(s);
  fake::capturing.erase(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  ++fake::n_sync;
  return fake::capturing.count(s) ? fake::fail(hipErrorStreamCaptureUnsupported) : hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
  *st = fake::capturing.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError(void) { const hipError_t e = fake::last; fake::last = hipSuccess; return e; }
const char* hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof *p);
  std::strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
}  // extern "C"
