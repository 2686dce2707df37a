/* The part of HIP's host interface that the workspace pool uses, on the CPU:
 * device memory is malloc'ed and may be limited, a stream runs only when the
 * test says so, and calls are counted. */
#pragma once
#include <stdint.h>
#include <stdlib.h>

#include <map>
#include <set>

#define __host__
#define __device__
#define __forceinline__ inline

enum hipError_t {
  hipSuccess = 0,
  hipErrorInvalidValue = 1,
  hipErrorOutOfMemory = 2,
  hipErrorInvalidHandle = 400,
  hipErrorNotReady = 600
};
struct FakeStream {
  long queued = 0, done = 0;  // work items
};
struct FakeEvent {
  FakeStream* s = nullptr;
  long at = 0;
};
typedef FakeStream* hipStream_t;
typedef FakeEvent* hipEvent_t;
#define hipStreamPerThread ((hipStream_t)2)
enum { hipEventDisableTiming = 2 };

struct Fake {
  size_t limit = SIZE_MAX, used = 0;
  std::map<void*, size_t> live;
  std::set<void*> freed_twice;
  long waits = 0, mallocs = 0, frees = 0;
  bool sync_fails = false;
  FakeStream per_thread;  // the calling thread's
};
inline Fake& fake() {
  static Fake f;
  return f;
}
inline FakeStream* real(hipStream_t s) { return s == hipStreamPerThread ? &fake().per_thread : s; }

inline const char* hipGetErrorString(hipError_t) { return "error"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
inline hipError_t hipMalloc(void** p, size_t n) {
  Fake& f = fake();
  if (f.used + n > f.limit) return hipErrorOutOfMemory;
  *p = malloc(16);
  f.live[*p] = n;
  f.used += n;
  ++f.mallocs;
  return hipSuccess;
}
template <typename T>
hipError_t hipMalloc(T** p, size_t n) {
  return hipMalloc(reinterpret_cast<void**>(p), n);
}
inline hipError_t hipFree(void* p) {
  Fake& f = fake();
  if (!p) return hipSuccess;
  auto it = f.live.find(p);
  if (it == f.live.end()) {
    f.freed_twice.insert(p);
    return hipErrorInvalidValue;
  }
  f.used -= it->second;
  f.live.erase(it);  // the address is not given out again
  ++f.frees;
  return hipSuccess;
}
inline hipError_t hipDeviceSynchronize() { return fake().sync_fails ? hipErrorInvalidHandle : hipSuccess; }
inline hipError_t hipStreamQuery(hipStream_t s) {
  return real(s)->done == real(s)->queued ? hipSuccess : hipErrorNotReady;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = new FakeEvent;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  e->s = real(s);
  e->at = e->s->queued;
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  if (e->s->done < e->at) e->s->done = e->at;
  return hipSuccess;
}
inline hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) {
  ++fake().waits;
  return hipSuccess;
}
