// hip_runtime.h -- the few HIP host calls of the transfer code, on the CPU: device
// memory is host memory, a stream runs its work at once. Streams know their
// device; what exists is counted, and a copy can be made to fail.
#pragma once

#include <atomic>
#include <cstddef>
#include <cstdlib>
#include <cstring>

enum hipError_t { hipSuccess = 0, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum { hipStreamNonBlocking = 1 };

namespace host_hip {
inline thread_local int device = 0;
inline std::atomic<int> streams{0}, created{0}, copies{0};
inline std::atomic<int> fail_copy{-1};  // the copy with this number fails
struct Stream {
  int dev;
};
}  // namespace host_hip
using hipStream_t = host_hip::Stream*;
using hipEvent_t = int*;

inline const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "success" : "failed on purpose"; }
inline hipError_t hipGetDevice(int* d) {
  *d = host_hip::device;
  return hipSuccess;
}
inline hipError_t hipSetDevice(int d) {
  host_hip::device = d;
  return hipSuccess;
}
inline hipError_t hipMalloc(void** p, size_t n) {
  *p = std::malloc(n);
  return *p ? hipSuccess : hipErrorUnknown;
}
inline hipError_t hipFree(void* p) {
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = new host_hip::Stream{host_hip::device};
  ++host_hip::streams;
  ++host_hip::created;
  return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s) {
  delete s;
  --host_hip::streams;
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t s) {
  if (s->dev != host_hip::device || host_hip::copies++ == host_hip::fail_copy) return hipErrorUnknown;
  std::memcpy(dst, src, n);
  return hipSuccess;
}
inline hipError_t hipMemcpy(void* dst, const void* src, size_t n, hipMemcpyKind) {
  std::memcpy(dst, src, n);
  return hipSuccess;
}
inline hipError_t hipEventCreate(hipEvent_t* e) {
  *e = new int(0);
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
