// Stand-in for the few runtime calls of host/column_copy.cpp, so that its host
// side runs and can be checked without a GPU.  A stream is a list of copies that
// are carried out as late as they may be: when an event behind them, or the
// stream, is waited for.
#ifndef TESTS_CPP_STAND_IN_HIP_RUNTIME_H_
#define TESTS_CPP_STAND_IN_HIP_RUNTIME_H_

#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <mutex>

enum hipError_t { hipSuccess = 0, hipErrorUnknown = 999, hipErrorNotReady = 600 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
constexpr unsigned hipEventDisableTiming = 2, hipHostMallocDefault = 0, hipHostMallocPortable = 1;

struct StandInCopy { void *to; const void *from; size_t bytes; };
struct StandInStream { std::deque<StandInCopy> queue; size_t done = 0; };
struct StandInEvent { StandInStream *stream = nullptr; size_t after = 0; };
using hipStream_t = StandInStream *;
using hipEvent_t = StandInEvent *;

struct StandInRuntime {
  std::mutex mutex;
  long copies_until_failure = -1;  // counts down; the copy that meets 0 fails
  size_t pinned = 0, most_pinned = 0, pinned_calls = 0;
  bool no_pinned = false;
};
inline StandInRuntime &Runtime() {
  static StandInRuntime r;
  return r;
}
inline void RunUpTo(hipStream_t s, size_t end) {
  for (; s->done < end; ++s->done) {
    const StandInCopy c = s->queue.front();
    s->queue.pop_front();
    std::memcpy(c.to, c.from, c.bytes);
  }
}
inline const char *hipGetErrorString(hipError_t) { return "stand-in error"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipMalloc(void *p, size_t n) {
  *static_cast<void **>(p) = std::malloc(n);
  return hipSuccess;
}
inline hipError_t hipFree(void *p) {
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  std::lock_guard<std::mutex> lock(Runtime().mutex);
  if (Runtime().no_pinned) return hipErrorUnknown;
  size_t *block = static_cast<size_t *>(std::malloc(n + 64));
  block[0] = n;
  *p = reinterpret_cast<char *>(block) + 64;
  Runtime().pinned += n;
  ++Runtime().pinned_calls;
  if (Runtime().pinned > Runtime().most_pinned) Runtime().most_pinned = Runtime().pinned;
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {
  std::lock_guard<std::mutex> lock(Runtime().mutex);
  size_t *block = reinterpret_cast<size_t *>(static_cast<char *>(p) - 64);
  Runtime().pinned -= block[0];
  std::free(block);
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void *to, const void *from, size_t bytes, hipMemcpyKind, hipStream_t s) {
  std::lock_guard<std::mutex> lock(Runtime().mutex);
  if (Runtime().copies_until_failure >= 0 && Runtime().copies_until_failure-- == 0) return hipErrorUnknown;
  s->queue.push_back({ to, from, bytes });
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  std::lock_guard<std::mutex> lock(Runtime().mutex);
  RunUpTo(s, s->done + s->queue.size());
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  *e = new StandInEvent;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  std::lock_guard<std::mutex> lock(Runtime().mutex);
  e->stream = s;
  e->after = s->done + s->queue.size();
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  std::lock_guard<std::mutex> lock(Runtime().mutex);
  if (e->stream) RunUpTo(e->stream, e->after);
  return hipSuccess;
}

#endif  // TESTS_CPP_STAND_IN_HIP_RUNTIME_H_
