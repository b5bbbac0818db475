// A HIP runtime on the host for the tests of the library's host code: device
// memory is malloc'd, filled with 0xa5, and every stream is a queue whose
// operations take place no sooner than the interface promises.  Streams do
// not order each other (they are created non-blocking); an operation of the
// null stream takes place after `sim_late` operations of the other streams,
// or when something waits for it.
#pragma once
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>

#define __host__
#define __device__
#define __align__(n) __attribute__((aligned(n)))
#define HIP_SYMBOL(x) (&x)

typedef int hipError_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum { hipStreamNonBlocking = 1, hipDeviceAttributeMultiprocessorCount = 0 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice };
struct int2 { int x, y; };

struct sim_stream {
  std::deque<std::function<void()>> q;
};
typedef sim_stream *hipStream_t;
typedef int *hipEvent_t;

inline sim_stream sim_null;
inline int sim_late = 0;                   // see above
inline int sim_after = 0;                  // operations seen since the null stream's oldest
inline long sim_alloc_left = 1l << 60;     // bytes that hipMalloc still gives

inline void sim_drain(sim_stream &s) {
  while (!s.q.empty()) {
    auto f = s.q.front();
    s.q.pop_front();
    f();
    if (&s != &sim_null && ++sim_after > sim_late) sim_drain(sim_null);
  }
  if (&s == &sim_null) sim_after = 0;
}
inline void sim_push(hipStream_t s, std::function<void()> f) {
  (s ? *s : sim_null).q.push_back(std::move(f));
  if (!s && sim_late == 0) sim_drain(sim_null);
}

inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
inline hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
inline hipError_t hipDeviceGetAttribute(int *v, int, int) { *v = 256; return hipSuccess; }
inline hipError_t hipMalloc(void **p, size_t n) {
  if ((long)n > sim_alloc_left) return hipErrorOutOfMemory;
  sim_alloc_left -= (long)n;
  *p = std::malloc(n);
  std::memset(*p, 0xa5, n);
  return hipSuccess;
}
inline hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
inline hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = new sim_stream; return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t s) { sim_drain(s ? *s : sim_null); return hipSuccess; }
inline hipError_t hipStreamDestroy(hipStream_t s) { delete s; return hipSuccess; }
inline hipError_t hipDeviceSynchronize() { return hipSuccess; }
inline hipError_t hipEventCreate(hipEvent_t *e) { *e = nullptr; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t s) { sim_drain(s ? *s : sim_null); return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
inline hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t s) {
  sim_push(s, [=] { std::memset(p, v, n); });
  return hipSuccess;
}
inline hipError_t hipMemset(void *p, int v, size_t n) { return hipMemsetAsync(p, v, n, nullptr); }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
  sim_push(st, [=] { std::memcpy(d, s, n); });
  return hipSuccess;
}
inline hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) {
  hipMemcpyAsync(d, s, n, k, nullptr);
  if (k != hipMemcpyDeviceToDevice) sim_drain(sim_null);   // these wait
  return hipSuccess;
}
inline hipError_t hipGetSymbolAddress(void **p, const void *s) { *p = const_cast<void *>(s); return hipSuccess; }
