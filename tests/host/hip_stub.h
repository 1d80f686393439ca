// The few HIP calls that gs_hostcopy.h makes, over plain host memory, with
// counters and failures on request: what a test of the copy on a CPU needs.
#pragma once
#include <stdint.h>
#include <stdlib.h>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
struct Stream {
  int syncs = 0;
};
typedef Stream* hipStream_t;
typedef int* hipEvent_t;
constexpr unsigned hipEventDisableTiming = 2, hipHostMallocDefault = 0;

inline int pinned = 0, pinnedMost = 0, mallocsLeft = 1 << 30, eventsLeft = 1 << 30, lastErrors = 0;

inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (mallocsLeft-- <= 0) return hipErrorOutOfMemory;
  size_t* q = (size_t*)malloc(n + 64);
  *q = n;
  pinned += (int)n;
  if (pinned > pinnedMost) pinnedMost = pinned;
  *p = (char*)q + 64;
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  size_t* q = (size_t*)((char*)p - 64);
  pinned -= (int)*q;
  free(q);
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  if (eventsLeft-- <= 0) return hipErrorUnknown;
  *e = new int(0);
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  ++*e;
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  s->syncs++;
  return hipSuccess;
}
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetLastError() {
  lastErrors++;
  return hipSuccess;
}
