// host/column_copy.cpp on the stand-in runtime (stand_in/hip/hip_runtime.h): what is
// put in comes out at the sizes where the copy changes form, and failures of the
// host leave the caller with a copy or an error, never with an abort.
#include <dlfcn.h>
#include <pthread.h>

#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <new>
#include <thread>
#include <vector>

#include "../../pvcriemannsolvers_amd/csrc/host/column_copy.hpp"
#include "../../pvcriemannsolvers_amd/csrc/host/common.hpp"

// operator new of this program fails once after `allocations_left` more calls
static std::atomic<long> allocations_left{ -1 };
void *operator new(size_t n) {
  if (allocations_left.load() >= 0 && allocations_left.fetch_sub(1) == 0) throw std::bad_alloc();
  if (void *p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

// Threads of this program begin only while the gate is open, or 3 s late.
static std::atomic<bool> gate_open{ true };
static std::atomic<int> forced_open{ 0 };
struct Start { void *(*run)(void *); void *arg; };
static void *AtTheGate(void *p) {
  const Start s = *static_cast<Start *>(p);
  std::free(p);
  for (int i = 0; i < 3000 && !gate_open.load(); ++i) std::this_thread::sleep_for(std::chrono::milliseconds(1));
  if (!gate_open.load()) forced_open.fetch_add(1);
  return s.run(s.arg);
}
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *attr, void *(*run)(void *), void *arg) {
  using Create = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
  static const Create create = reinterpret_cast<Create>(dlsym(RTLD_NEXT, "pthread_create"));
  Start *s = static_cast<Start *>(std::malloc(sizeof(Start)));
  *s = { run, arg };
  return create(t, attr, AtTheGate, s);
}

namespace mcfd {
std::string &LastError() {
  thread_local std::string e;
  return e;
}
}  // namespace mcfd

namespace {

constexpr size_t kMiB = size_t(1) << 20;

std::vector<char> Pattern(size_t n, unsigned seed) {
  std::vector<char> v(n);
  for (size_t i = 0; i < n; ++i) v[i] = (char)((i * 2654435761u + seed) >> 13);
  return v;
}

struct Handle {
  mcfd::ColumnCopy copy;
  StandInStream stream;
  std::vector<char> device;
  explicit Handle(size_t n) : device(n) { copy.Reserve(n); }
  ~Handle() { (void)hipStreamSynchronize(&stream); }
  bool In(const std::vector<char> &host) {
    std::lock_guard<std::mutex> lock(copy.mutex);
    copy.ToDevice(device.data(), host.data(), host.size(), &stream);
    copy.Wait(&stream);
    return std::memcmp(device.data(), host.data(), host.size()) == 0;
  }
  bool Out() {
    std::vector<char> host(device.size(), 0);
    std::lock_guard<std::mutex> lock(copy.mutex);
    copy.ToHost(host.data(), device.data(), host.size(), &stream);
    return host == device;
  }
};

const size_t kSizes[] = { 8, 2 * kMiB - 8, 2 * kMiB, 2 * kMiB + 8, 5 * kMiB + 24, 16 * kMiB, 17 * kMiB + 40,
                          32 * kMiB - 8, 32 * kMiB, 32 * kMiB + 8, 67 * kMiB + 16 };

bool RoundTrips() {
  for (size_t n : kSizes) {
    Handle h(n);
    for (unsigned seed = 0; seed < 2; ++seed)
      if (!h.In(Pattern(n, seed)) || !h.Out()) return false;
  }
  return true;
}

// Memory runs out while the copy's threads are started, at every allocation of it.
bool NoMemoryForThreads() {
  for (size_t n : { 5 * kMiB, 40 * kMiB }) {
    Handle h(n);
    const std::vector<char> host = Pattern(n, 3);
    std::vector<char> back(n);
    for (long k = 0; k < 12; ++k) {
      std::lock_guard<std::mutex> lock(h.copy.mutex);
      bool in = false, out = false;
      allocations_left = k;
      try {
        h.copy.ToDevice(h.device.data(), host.data(), n, &h.stream);
        in = true;
      } catch (std::bad_alloc const &) {
      }
      allocations_left = -1;
      (void)hipStreamSynchronize(&h.stream);
      if (in && h.device != host) return false;
      h.device = host;
      allocations_left = k;
      try {
        h.copy.ToHost(back.data(), h.device.data(), n, &h.stream);
        out = true;
      } catch (std::bad_alloc const &) {
      }
      allocations_left = -1;
      if (out && back != host) return false;
      back.assign(n, 0);
    }
  }
  return true;
}

// A copy that fails on its way leaves copies to and from the slots in flight; what
// follows it on the same handle is whole all the same.
bool CopiesAfterAFailure() {
  for (size_t n : { 7 * kMiB, 40 * kMiB }) {
    Handle h(n);
    for (long k : { 0, 1, 3, 9, 20 }) {
      for (bool in : { false, true }) {
        std::vector<char> host = Pattern(n, (unsigned)k), other = Pattern(n, (unsigned)k + 1);
        Runtime().copies_until_failure = k;
        bool failed = false;
        try {
          std::lock_guard<std::mutex> lock(h.copy.mutex);
          if (in) h.copy.ToDevice(h.device.data(), other.data(), n, &h.stream);
          else h.copy.ToHost(other.data(), h.device.data(), n, &h.stream);
        } catch (mcfd::Failure const &) {
          failed = true;
        }
        if (failed != (Runtime().copies_until_failure == -1)) return false;
        Runtime().copies_until_failure = -1;
        if (!h.In(host) || !h.Out()) return false;
      }
    }
  }
  return true;
}

// No thread of a copy begins before the copy returns: processors that are busy.
bool ThreadsThatBeginLate() {
  for (size_t n : { 3 * kMiB, 40 * kMiB }) {
    Handle h(n);
    gate_open = false;
    bool ok = true;
    for (unsigned seed = 0; seed < 4; ++seed) ok = ok && h.In(Pattern(n, seed)) && h.Out();
    ok = ok && forced_open.load() == 0;
    gate_open = true;
    if (!ok || !h.In(Pattern(n, 9)) || !h.Out()) return false;
  }
  return true;
}

// The rings belong to all handles: no more than four, none where there is no
// handle, large enough for the largest, and each handle's columns its own when
// all copy at once.
bool RingsOfAllHandles() {
  if (Runtime().pinned != 0) return false;
  Runtime().pinned_calls = Runtime().most_pinned = 0;
  {
    std::vector<std::unique_ptr<Handle>> handles;
    for (int i = 0; i < 12; ++i) handles.push_back(std::make_unique<Handle>(5 * kMiB));
    if (Runtime().pinned_calls > 4 || Runtime().most_pinned > 20 * kMiB) return false;
    handles.push_back(std::make_unique<Handle>(70 * kMiB));
    const size_t calls = Runtime().pinned_calls, bytes = Runtime().pinned;
    if (calls != 5 || bytes > 47 * kMiB) return false;
    std::atomic<int> wrong{ 0 };
    std::vector<std::thread> users;
    for (size_t i = 0; i < handles.size(); ++i)
      users.emplace_back([&, i] {
        for (unsigned k = 0; k < 3; ++k)
          if (!handles[i]->In(Pattern(handles[i]->device.size(), (unsigned)(7 * i) + k)) || !handles[i]->Out()) ++wrong;
      });
    for (auto &u : users) u.join();
    if (wrong.load() || Runtime().pinned_calls != calls) return false;
    handles.resize(2);
    if (Runtime().pinned > bytes - 10 * kMiB || !handles[1]->Out()) return false;
  }
  if (Runtime().pinned != 0) return false;
  Runtime().no_pinned = true;
  const bool direct = [] {
    Handle h(33 * kMiB);
    return h.In(Pattern(33 * kMiB, 1)) && h.Out();
  }();
  Runtime().no_pinned = false;
  return direct;
}

}  // namespace

int main(int argc, char **argv) {
  const struct { const char *name; bool (*run)(); } tests[] = { { "round_trips", RoundTrips },
                                                                { "no_memory_for_threads", NoMemoryForThreads },
                                                                { "copies_after_a_failure", CopiesAfterAFailure },
                                                                { "threads_that_begin_late", ThreadsThatBeginLate },
                                                                { "rings_of_all_handles", RingsOfAllHandles } };
  for (auto const &t : tests) {
    if (argc > 1 && std::strcmp(argv[1], t.name) != 0) continue;
    const bool ok = t.run();
    std::printf("%s %s\n", ok ? "PASS" : "FAIL", t.name);
    if (!ok) return 1;
  }
  return 0;
}
