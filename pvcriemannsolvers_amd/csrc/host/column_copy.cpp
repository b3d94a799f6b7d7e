#include "column_copy.hpp"

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <exception>
#include <thread>
#include <vector>

#include "common.hpp"

namespace mcfd {
namespace {

// Where the ring takes over.  Measured, us direct -> ring, to the host into pages
// just handed out and into used ones: 2.6 MB 640 -> 350 and 167 -> 131, 4.1 MB
// 1030 -> 424 and 246 -> 194, 11.8 MB 1550 -> 568 and 690 -> 432, 130 MB 13490 -> 3550
// and 12320 -> 3600; below 2 MB nothing is left to share.  To the device: 4.1 MB
// 150 -> 215, 11.8 MB 370 -> 466, 32 MB 965 -> 924, 65 MB 2200 -> 1770.
constexpr size_t kLeastToHost = size_t(2) << 20, kLeastToDevice = size_t(32) << 20;
// One copy of a chunk costs the caller about 8 us of launches: chunks of 256 KB
// take 326 us for 4.1 MB, of 1 MB 194.
constexpr size_t kLeastChunk = size_t(1) << 20, kMostChunk = size_t(2) << 20;

// Host threads that run `work` beside the caller; joined on every way out.
class Crew {
 public:
  template <class Work>
  Crew(int n, Work const &work) {
    try {
      threads_.reserve(n);
      for (int i = 0; i < n; ++i) threads_.emplace_back(work);
    } catch (std::exception const &) {  // no threads or no memory left: fewer than wished for
    }
  }
  ~Crew() {
    for (auto &t : threads_) t.join();
  }
  bool empty() const { return threads_.empty(); }

 private:
  std::vector<std::thread> threads_;
};

// Sets the flag unless the scope is left normally.
struct StopOnFailure {
  std::atomic<bool> &stop;
  bool done = false;
  ~StopOnFailure() {
    if (!done) stop.store(true);
  }
};

}  // namespace

size_t ColumnCopy::Chunk(size_t bytes) {
  const size_t even = (bytes / kSlots + 4095) & ~size_t(4095);
  return std::min(kMostChunk, std::max(kLeastChunk, even));
}

bool ColumnCopy::Ring(size_t bytes, size_t least) const {
  const size_t chunk = Chunk(bytes);
  return pinned_ && bytes >= least && chunk <= slot_ && (bytes + chunk - 1) / chunk <= most_;
}

void ColumnCopy::Reserve(size_t bytes) {
  if (pinned_ || bytes < kLeastToHost) return;
  for (auto &e : events_) Check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "column copy event");
  const size_t slot = Chunk(bytes), chunks = (bytes + slot - 1) / slot, slots = std::min<size_t>(chunks, kSlots);
  void *p = nullptr;
  if (hipHostMalloc(&p, slot * slots, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    return;
  }
  pinned_ = static_cast<char *>(p);
  slot_ = slot;
  most_ = slots < kSlots ? slots : SIZE_MAX;
}

ColumnCopy::~ColumnCopy() {
  if (pinned_) (void)hipHostFree(pinned_);
  for (auto &e : events_)
    if (e) (void)hipEventDestroy(e);
}

void ColumnCopy::Settle() {
  if (!busy_) return;
  Check(hipStreamSynchronize(busy_), "column copy sync");
  busy_ = nullptr;
}

void ColumnCopy::ToHost(void *host, const void *device, size_t bytes, hipStream_t stream) {
  if (!Ring(bytes, kLeastToHost)) {
    Check(hipMemcpyAsync(host, device, bytes, hipMemcpyDeviceToHost, stream), "column to host");
    Check(hipStreamSynchronize(stream), "column to host sync");
    return;
  }
  Settle();
  busy_ = stream;
  const size_t chunk = Chunk(bytes);
  const int64_t n = (int64_t)((bytes + chunk - 1) / chunk);
  auto size = [&](int64_t c) { return std::min(chunk, bytes - size_t(c) * chunk); };
  std::atomic<int64_t> next{ 0 }, filled{ 0 };  // the next chunk to take; chunks that are in their slots
  std::atomic<int64_t> taken[kSlots];           // the last chunk copied out of the slot
  for (auto &t : taken) t.store(-1);
  std::atomic<bool> stop{ false };
  auto work = [&] {
    for (int64_t c; (c = next.fetch_add(1)) < n;) {
      while (filled.load(std::memory_order_acquire) <= c) {
        if (stop.load()) return;
        std::this_thread::yield();
      }
      std::memcpy(static_cast<char *>(host) + size_t(c) * chunk, pinned_ + size_t(c % kSlots) * slot_, size(c));
      taken[c % kSlots].store(c, std::memory_order_release);
    }
  };
  int64_t issued = 0;
  auto issue = [&] {
    while (issued < n &&
           (issued < kSlots || taken[issued % kSlots].load(std::memory_order_acquire) == issued - kSlots)) {
      const int s = (int)(issued % kSlots);
      Check(hipMemcpyAsync(pinned_ + size_t(s) * slot_, static_cast<const char *>(device) + size_t(issued) * chunk,
                           size(issued), hipMemcpyDeviceToHost, stream), "column to host");
      Check(hipEventRecord(events_[s], stream), "column to host event");
      ++issued;
    }
  };
  issue();  // the first copies run while the threads start
  {
    Crew crew((int)std::min<int64_t>(kThreads, n), work);
    StopOnFailure guard{ stop };
    for (int64_t c = 0; c < n; ++c) {
      while (issued <= c) {  // all slots wait to be emptied
        if (crew.empty()) break;
        issue();
        std::this_thread::yield();
      }
      if (crew.empty()) break;
      Check(hipEventSynchronize(events_[c % kSlots]), "column to host sync");
      filled.store(c + 1, std::memory_order_release);
      issue();
    }
    guard.done = true;
    if (crew.empty()) {
      Check(hipMemcpyAsync(host, device, bytes, hipMemcpyDeviceToHost, stream), "column to host");
      Check(hipStreamSynchronize(stream), "column to host sync");
    }
  }
  busy_ = nullptr;
}

void ColumnCopy::ToDevice(void *device, const void *host, size_t bytes, hipStream_t stream) {
  if (!Ring(bytes, kLeastToDevice)) {
    Check(hipMemcpyAsync(device, host, bytes, hipMemcpyHostToDevice, stream), "column to device");
    return;
  }
  Settle();
  busy_ = stream;
  const size_t chunk = Chunk(bytes);
  const int64_t n = (int64_t)((bytes + chunk - 1) / chunk);
  auto size = [&](int64_t c) { return std::min(chunk, bytes - size_t(c) * chunk); };
  std::atomic<int64_t> next{ 0 }, drained{ 0 };  // the next chunk to take; chunks whose slots are free again
  std::atomic<int64_t> put[kSlots];              // the last chunk copied into the slot
  for (auto &p : put) p.store(-1);
  std::atomic<bool> stop{ false };
  auto work = [&] {
    for (int64_t c; (c = next.fetch_add(1)) < n;) {
      while (drained.load(std::memory_order_acquire) <= c - kSlots) {
        if (stop.load()) return;
        std::this_thread::yield();
      }
      std::memcpy(pinned_ + size_t(c % kSlots) * slot_, static_cast<const char *>(host) + size_t(c) * chunk, size(c));
      put[c % kSlots].store(c, std::memory_order_release);
    }
  };
  {
    Crew crew((int)std::min<int64_t>(kThreads, n), work);
    StopOnFailure guard{ stop };
    int64_t done = 0;
    for (int64_t c = 0; c < n && !crew.empty(); ++c) {
      // half of the slots on their way to the device, the other half being filled
      for (; c - done >= kSlots / 2; ++done) {
        Check(hipEventSynchronize(events_[done % kSlots]), "column to device sync");
        drained.store(done + 1, std::memory_order_release);
      }
      while (put[c % kSlots].load(std::memory_order_acquire) != c) std::this_thread::yield();
      const int s = (int)(c % kSlots);
      Check(hipMemcpyAsync(static_cast<char *>(device) + size_t(c) * chunk, pinned_ + size_t(s) * slot_, size(c),
                           hipMemcpyHostToDevice, stream), "column to device");
      Check(hipEventRecord(events_[s], stream), "column to device event");
    }
    guard.done = true;
    if (crew.empty())
      Check(hipMemcpyAsync(device, host, bytes, hipMemcpyHostToDevice, stream), "column to device");
  }
}

}  // namespace mcfd
