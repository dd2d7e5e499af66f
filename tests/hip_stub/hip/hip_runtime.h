// A stand-in for the HIP runtime, for CPU tests of host code and of device
// functions that are plain arithmetic.  Copies on a stream are put off until
// something waits for them, as late as a real device may run them, so a
// missing wait shows as wrong bytes.  Failures are set through stub::.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <stdexcept>

#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))
#define __builtin_amdgcn_rcp(x) (1.0 / (x))
using std::fabs;
using std::fmax;
using std::signbit;

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2, hipMemcpyDeviceToDevice = 3 };
enum hipMemoryType { hipMemoryTypeHost = 0, hipMemoryTypeDevice = 1, hipMemoryTypeManaged = 2, hipMemoryTypeUnregistered = 3 };
struct hipPointerAttribute_t {
  hipMemoryType type;
};
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;
enum hipDeviceAttribute_t { hipDeviceAttributeMultiprocessorCount };

namespace stub {
struct Copy {
  void *dst;
  const void *src;
  size_t n;
};
struct Stream {
  std::deque<Copy> todo;
  uint64_t enqueued = 0, done = 0;
  std::mutex mu;
  void run_to(uint64_t upto) {
    std::lock_guard<std::mutex> g(mu);
    while (done < upto) {
      std::memcpy(todo.front().dst, todo.front().src, todo.front().n);
      todo.pop_front();
      done++;
    }
  }
};
struct Event {
  Stream *s = nullptr;
  uint64_t at = 0;
};
inline std::mutex mu;
inline int pinned_left = -1;  // hipHostMalloc calls that still succeed (-1: all)
inline int pinned_live = 0;
inline std::map<const char *, size_t> pinned;
inline int copies_left = -1;  // hipMemcpyAsync calls that still succeed
inline bool copies_throw = false;
inline bool is_pinned(const void *p) {
  std::lock_guard<std::mutex> g(mu);
  auto it = pinned.upper_bound(static_cast<const char *>(p));
  return it != pinned.begin() && (--it, static_cast<const char *>(p) < it->first + it->second);
}
inline bool take(int &left) {
  std::lock_guard<std::mutex> g(mu);
  if (left == 0) return false;
  if (left > 0) left--;
  return true;
}
}  // namespace stub

using hipStream_t = stub::Stream *;
using hipEvent_t = stub::Event *;

inline const char *hipGetErrorString(hipError_t) { return "stub error"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
template <class T>
hipError_t hipMalloc(T **p, size_t n) {
  *p = static_cast<T *>(std::malloc(n));
  return hipSuccess;
}
inline hipError_t hipFree(void *p) {
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipMemGetInfo(size_t *f, size_t *t) {
  *f = *t = (size_t)1 << 30;
  return hipSuccess;
}
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  if (!stub::take(stub::pinned_left)) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  std::lock_guard<std::mutex> g(stub::mu);
  stub::pinned_live++;
  stub::pinned[static_cast<char *>(*p)] = n;
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {
  std::lock_guard<std::mutex> g(stub::mu);
  stub::pinned.erase(static_cast<char *>(p));
  std::free(p);
  stub::pinned_live--;
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  uint64_t n;
  {
    std::lock_guard<std::mutex> g(s->mu);
    n = s->enqueued;
  }
  s->run_to(n);
  return hipSuccess;
}
// A copy from or to pageable host memory has read or written it on return.
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind kind, hipStream_t st) {
  if (!d || !s) return hipErrorInvalidValue;
  if (!stub::take(stub::copies_left)) {
    if (stub::copies_throw) throw std::runtime_error("planted");
    return hipErrorInvalidValue;
  }
  {
    std::lock_guard<std::mutex> g(st->mu);
    st->todo.push_back({d, s, n});
    st->enqueued++;
  }
  if (!stub::is_pinned(kind == hipMemcpyHostToDevice ? s : d)) return hipStreamSynchronize(st);
  return hipSuccess;
}
inline hipError_t hipEventCreate(hipEvent_t *e) {
  *e = new stub::Event;
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  std::lock_guard<std::mutex> g(s->mu);
  e->s = s;
  e->at = s->enqueued;
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  if (e->s) e->s->run_to(e->at);
  return hipSuccess;
}
inline hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 0;
  return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) {
  a->type = hipMemoryTypeUnregistered;
  return hipSuccess;
}
