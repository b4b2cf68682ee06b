// The few HIP calls of fd2_hostcopy.h on the CPU, for tests: device memory is
// host memory, and a stream's copies run only when the stream or one of their
// events is waited for.  Unlike the runtime's own, hipHostFree and
// hipEventDestroy wait for nothing: freeing memory that a queued copy still
// needs, or destroying an event that is still to be reached, counts in
// `faults`.
#pragma once
#include <stdlib.h>
#include <string.h>

#include <deque>
#include <mutex>

enum hipError_t { hipSuccess = 0, hipErrorUnknown = 1 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

namespace hipstub {
struct Event {
  bool reached = true;
};
struct Op {  // a copy, or the mark of an event
  char* dst;
  const char* src;
  size_t n;
  Event* event;
};
inline std::mutex mu;
inline std::deque<Op> queue;  // one stream
inline int faults = 0, ring_frees = 0;
inline bool no_pinned = false;  // hipHostMalloc fails
inline const char* ring = nullptr;
inline size_t ring_bytes = 0;
inline void step() {
  const Op op = queue.front();
  queue.pop_front();
  if (op.event)
    op.event->reached = true;
  else
    memcpy(op.dst, op.src, op.n);
}
inline bool in_ring(const char* p) { return ring && p >= ring && p < ring + ring_bytes; }
}  // namespace hipstub

typedef int hipStream_t;
typedef hipstub::Event* hipEvent_t;

inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (hipstub::no_pinned) return hipErrorUnknown;
  *p = malloc(n);
  hipstub::ring = static_cast<char*>(*p);
  hipstub::ring_bytes = n;
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  std::lock_guard<std::mutex> l(hipstub::mu);
  for (const hipstub::Op& op : hipstub::queue)
    if (!op.event && (hipstub::in_ring(op.dst) || hipstub::in_ring(op.src))) ++hipstub::faults;
  ++hipstub::ring_frees;
  hipstub::ring = nullptr;
  while (!hipstub::queue.empty()) hipstub::step();  // so that the test itself stays sound
  free(p);
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = new hipstub::Event;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  std::lock_guard<std::mutex> l(hipstub::mu);
  if (!e->reached) {
    ++hipstub::faults;
    while (!hipstub::queue.empty()) hipstub::step();
  }
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  std::lock_guard<std::mutex> l(hipstub::mu);
  e->reached = false;
  hipstub::queue.push_back({nullptr, nullptr, 0, e});
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  std::lock_guard<std::mutex> l(hipstub::mu);
  while (!e->reached) hipstub::step();
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
  std::lock_guard<std::mutex> l(hipstub::mu);
  hipstub::queue.push_back({static_cast<char*>(dst), static_cast<const char*>(src), n, nullptr});
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) {
  std::lock_guard<std::mutex> l(hipstub::mu);
  while (!hipstub::queue.empty()) hipstub::step();
  return hipSuccess;
}
