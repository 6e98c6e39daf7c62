// The few HIP calls of staging.hpp on the CPU, as late as a device may be: a
// copy put on a stream moves its bytes only when the stream (or an event
// after it) is waited for.  Any call can be made to fail; host memory freed
// while a copy still uses it, or put to another use, shows as wrong bytes or a
// report.
#pragma once
#include <cstddef>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <mutex>
#include <set>

enum hipError_t { hipSuccess = 0, hipErrorInvalidDevice = 101, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
constexpr unsigned hipHostMallocPortable = 1, hipEventDisableTiming = 2;

namespace stub {
struct Copy {
  void* to;
  const void* from;
  size_t n;
};
struct Stream {
  std::deque<Copy> q;
  size_t done = 0;  // copies ever finished
};
struct Event {
  Stream* s = nullptr;
  size_t upto = 0;
};
inline std::mutex mu;
inline long copies = 0, fail_copy = -1;        // the copy (from 0) that fails
inline long allocs = 0, live = 0, fail_alloc = -1;
inline std::set<Stream*> streams;
inline bool used(const void* p, size_t n) {  // by a copy not yet made
  std::lock_guard<std::mutex> l(mu);
  const char *a = (const char*)p, *b = a + n;
  for (auto* s : streams)
    for (auto& c : s->q)
      for (const char* x : {(const char*)c.to, (const char*)c.from})
        if (x < b && x + c.n > a) return true;
  return false;
}
inline void run(Stream* s, size_t upto) {
  while (s->done < upto && !s->q.empty()) {
    std::memcpy(s->q.front().to, s->q.front().from, s->q.front().n);
    s->q.pop_front();
    ++s->done;
  }
}
}  // namespace stub
typedef stub::Stream* hipStream_t;
typedef stub::Event* hipEvent_t;

inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  std::lock_guard<std::mutex> l(stub::mu);
  if (stub::allocs++ == stub::fail_alloc || stub::fail_alloc == -2) return hipErrorUnknown;
  *p = std::malloc(n);
  ++stub::live;
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  std::lock_guard<std::mutex> l(stub::mu);
  std::free(p);
  --stub::live;
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind,
                                 hipStream_t s) {
  std::lock_guard<std::mutex> l(stub::mu);
  stub::streams.insert(s);
  if (stub::copies++ == stub::fail_copy) return hipErrorUnknown;
  s->q.push_back({to, from, n});
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  std::lock_guard<std::mutex> l(stub::mu);
  stub::run(s, s->done + s->q.size());
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = new stub::Event;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  std::lock_guard<std::mutex> l(stub::mu);
  e->s = s;
  e->upto = s->done + s->q.size();
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  std::lock_guard<std::mutex> l(stub::mu);
  if (e->s) stub::run(e->s, e->upto);
  return hipSuccess;
}
