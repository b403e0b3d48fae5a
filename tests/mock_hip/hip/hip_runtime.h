// A host-only stand-in for the HIP runtime calls of csrc/ctx.hip.  "Device"
// memory is host memory.  Streams hold what is enqueued until something waits
// for it, so that all that may be in flight is.  mock::fail_copy makes the
// n-th asynchronous copy from now fail (0: the next one).
#pragma once
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <set>
#include <string>
#include <system_error>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorNotReady, hipErrorUnknown };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice };

namespace mock {
struct Event;
struct Op {
  std::function<void()> run;    // empty for the two below
  Event* record = nullptr;
  Event* wait = nullptr;
  int generation = 0;
};
struct Stream {
  std::deque<Op> ops;
};
struct Event {
  Stream* on = nullptr;
  int recorded = 0, done = 0;   // generations
};
inline std::set<Stream*>& streams() {
  static std::set<Stream*> s;
  return s;
}
inline int fail_copy = -1;

// run a stream's work, up to generation g of event e if given
inline void drain(Stream* s, Event* e = nullptr, int g = 0) {
  while (!s->ops.empty() && !(e && e->done >= g)) {
    Op op = s->ops.front();
    s->ops.pop_front();
    if (op.wait && op.wait->on) drain(op.wait->on, op.wait, op.generation);
    if (op.run) op.run();
    if (op.record) op.record->done = std::max(op.record->done, op.generation);
  }
}
}  // namespace mock

using hipStream_t = mock::Stream*;
using hipEvent_t = mock::Event*;
struct hipDeviceProp_t {
  int multiProcessorCount = 0;
};
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 0, hipStreamNonBlocking = 0;

inline const char* hipGetErrorString(hipError_t) { return "mock error"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipMemGetInfo(size_t* f, size_t* t) { return *f = *t = size_t(1) << 30, hipSuccess; }
inline hipError_t hipGetDeviceProperties(hipDeviceProp_t*, int) { return hipSuccess; }

inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  mock::streams().insert(*s = new mock::Stream());
  return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s) {
  mock::drain(s);
  mock::streams().erase(s);
  delete s;
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) { return mock::drain(s), hipSuccess; }
inline hipError_t hipDeviceSynchronize() {
  for (mock::Stream* s : mock::streams()) mock::drain(s);
  return hipSuccess;
}

template <class T>
hipError_t hipMalloc(T** p, size_t n) {
  return (*p = (T*)std::malloc(n)) ? hipSuccess : hipErrorUnknown;
}
inline hipError_t hipFree(void* p) { return hipDeviceSynchronize(), std::free(p), hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  return (*p = std::malloc(n)) ? hipSuccess : hipErrorUnknown;
}
inline hipError_t hipHostFree(void* p) { return hipDeviceSynchronize(), std::free(p), hipSuccess; }

inline hipError_t hipEventCreate(hipEvent_t* e) { return *e = new mock::Event(), hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
inline hipError_t hipEventDestroy(hipEvent_t e) {
  hipDeviceSynchronize();
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0, hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  e->on = s;
  s->ops.push_back({{}, e, nullptr, ++e->recorded});
  return hipSuccess;
}
inline hipError_t hipEventQuery(hipEvent_t e) {
  return e->done == e->recorded ? hipSuccess : hipErrorNotReady;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  if (e->on) mock::drain(e->on, e, e->recorded);
  return hipSuccess;
}
inline hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  if (e->on) s->ops.push_back({{}, nullptr, e, e->recorded});
  return hipSuccess;
}

inline hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w,
                                   size_t h, hipMemcpyKind, hipStream_t st) {
  if (mock::fail_copy >= 0 && mock::fail_copy-- == 0) return hipErrorUnknown;
  st->ops.push_back({[=] {
    for (size_t j = 0; j < h; ++j) std::memcpy((char*)d + j * dp, (const char*)s + j * sp, w);
  }});
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k,
                                 hipStream_t st) {
  return hipMemcpy2DAsync(d, n, s, n, n, 1, k, st);
}
inline hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  hipDeviceSynchronize();
  std::memcpy(d, s, n);
  return hipSuccess;
}
