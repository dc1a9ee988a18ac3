// A runtime of two devices in host memory, for tests of host code without a
// GPU: copies run at once, an event belongs to the device that was current when
// it was created and can be recorded on that device's streams only.
#pragma once
#include <stddef.h>
#include <string.h>

#include <condition_variable>
#include <mutex>
#include <set>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorInvalidHandle = 400 };
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered, hipMemoryTypeHost, hipMemoryTypeDevice, hipMemoryTypeManaged };
struct hipPointerAttribute_t { hipMemoryType type; };
struct FakeStream { int device; };
struct FakeEvent { int device; };
typedef FakeStream* hipStream_t;
typedef FakeEvent* hipEvent_t;
typedef int hipDevice_t;
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

namespace fake {
inline thread_local int device = 0;
inline std::mutex mu;
inline std::set<void*> pinned;             // from hipHostMalloc
inline size_t pinned_peak = 0;             // the most of them at once
inline int meet = 0, met = 0;              // copies wait until `meet` have begun (0: none waits)
inline std::condition_variable all_met;
inline void* known = nullptr;              // a pointer the runtime knows
inline hipMemoryType known_type = hipMemoryTypeDevice;
inline int records_left = -1;              // event records before they fail (-1: never)
inline int live_events = 0;
struct Copy { void* dst; size_t n; };
inline Copy last{nullptr, 0};              // the last transfer
}  // namespace fake

inline hipError_t hipGetDevice(int* d) { *d = fake::device; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { fake::device = d; return hipSuccess; }
inline hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) { *d = s->device; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  std::lock_guard<std::mutex> lk(fake::mu);
  *p = ::operator new(n);
  fake::pinned.insert(*p);
  if (fake::pinned.size() > fake::pinned_peak) fake::pinned_peak = fake::pinned.size();
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  std::lock_guard<std::mutex> lk(fake::mu);
  fake::pinned.erase(p);
  ::operator delete(p);
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  ++fake::live_events;
  *e = new FakeEvent{fake::device};
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { --fake::live_events; delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (fake::records_left == 0) return hipErrorInvalidHandle;
  if (fake::records_left > 0) --fake::records_left;
  return e->device == s->device ? hipSuccess : hipErrorInvalidHandle;
}
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
  memcpy(dst, src, n);
  std::unique_lock<std::mutex> lk(fake::mu);
  fake::last = {dst, n};
  if (fake::met < fake::meet && ++fake::met == fake::meet) fake::all_met.notify_all();
  fake::all_met.wait(lk, [] { return fake::met >= fake::meet; });
  return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  if (p != fake::known) return hipErrorInvalidValue;
  a->type = fake::known_type;
  return hipSuccess;
}
