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

constexpr int kMostRings = 4;

size_t Chunk(size_t bytes) {
  const size_t even = (bytes / ColumnCopy::kSlots + 4095) & ~size_t(4095);
  return std::min(kMostChunk, std::max(kLeastChunk, even));
}
// Bytes of the ring that a column of `bytes` goes through.
size_t RingBytes(size_t bytes) {
  const size_t chunk = Chunk(bytes), chunks = (bytes + chunk - 1) / chunk;
  return chunk * std::min<size_t>(chunks, ColumnCopy::kSlots);
}

// The process's rings.  Never destroyed itself: the last user frees the rings, and
// a handle that outlives main's statics still finds it.
class Rings {
 public:
  static Rings &Get() {
    static Rings *rings = new Rings;
    return *rings;
  }
  // One more user with columns of up to `bytes`: one ring more, up to kMostRings,
  // or a larger one in place of the smallest that is not lent.
  void Enter(size_t bytes) {
    auto ring = std::make_unique<ColumnCopy::Ring>();
    std::lock_guard<std::mutex> lock(mutex_);
    idle_.reserve(kMostRings);
    ++users_;
    const size_t need = RingBytes(bytes);
    if (idle_.size() + lent_ >= (size_t)std::min(users_, kMostRings)) {
      for (auto const &r : idle_)
        if (r->bytes >= need) return;
      if (idle_.empty()) return;
      Free(Smallest());
    }
    void *p = nullptr;
    if (hipHostMalloc(&p, need, hipHostMallocPortable) != hipSuccess) {
      (void)hipGetLastError();
      return;
    }
    ring->pinned = static_cast<char *>(p);
    ring->bytes = need;
    idle_.insert(idle_.begin(), std::move(ring));  // behind those whose pages are known
  }
  void Leave() {
    std::lock_guard<std::mutex> lock(mutex_);
    --users_;
    while (!idle_.empty() && idle_.size() + lent_ > (size_t)users_) Free(Smallest());
  }
  // The ring used last of those that are large enough, or null.
  ColumnCopy::Ring *Lend(size_t bytes) {
    std::lock_guard<std::mutex> lock(mutex_);
    const size_t need = RingBytes(bytes);
    for (size_t i = idle_.size(); i-- > 0;) {
      if (idle_[i]->bytes < need) continue;
      ColumnCopy::Ring *ring = idle_[i].release();
      idle_.erase(idle_.begin() + (long)i);
      ++lent_;
      return ring;
    }
    return nullptr;
  }
  void Return(ColumnCopy::Ring *ring) {
    std::lock_guard<std::mutex> lock(mutex_);
    --lent_;
    idle_.emplace_back(ring);
  }

 private:
  size_t Smallest() const {
    size_t at = 0;
    for (size_t i = 1; i < idle_.size(); ++i)
      if (idle_[i]->bytes < idle_[at]->bytes) at = i;
    return at;
  }
  void Free(size_t at) {
    (void)hipHostFree(idle_[at]->pinned);
    idle_.erase(idle_.begin() + (long)at);
  }
  std::mutex mutex_;
  std::vector<std::unique_ptr<ColumnCopy::Ring>> idle_;  // the last used at the end
  size_t lent_ = 0;
  int users_ = 0;
};

}  // namespace

// One column's chunks, claimed in order by whoever is free.  A thread that begins
// after the call has returned finds none left and touches nothing else.
struct ColumnCopy::Job {
  char *host, *pinned;
  size_t bytes, chunk;
  int64_t n;
  bool to_host;
  std::atomic<int64_t> next{ 0 };    // to be claimed
  std::atomic<int64_t> limit{ 0 };   // claimed only below: the slot is filled, or free
  std::atomic<int64_t> copied{ 0 };
  std::atomic<int64_t> last[kSlots];  // the chunk copied last from or to the slot
  std::atomic<bool> begun[kThreads] = {};
  std::atomic<bool> ended[kThreads] = {};
  std::atomic<int> at_work{ 0 };

  Job(void *h, Ring const &ring, size_t size, bool out)
      : host(static_cast<char *>(h)), pinned(ring.pinned), bytes(size), chunk(Chunk(size)),
        n((int64_t)((size + chunk - 1) / chunk)), to_host(out) {
    for (auto &l : last) l.store(-1);
  }
  size_t Size(int64_t c) const { return std::min(chunk, bytes - size_t(c) * chunk); }
  char *Slot(int64_t c) const { return pinned + size_t(c % kSlots) * chunk; }
  bool Holds(int64_t c) const { return last[c % kSlots].load(std::memory_order_acquire) == c; }
  // Copies the next chunk, if it can be claimed.
  bool Step() {
    int64_t c = next.load();
    do {
      if (c >= limit.load(std::memory_order_acquire)) return false;
    } while (!next.compare_exchange_weak(c, c + 1));
    char *const at = host + size_t(c) * chunk;
    if (to_host) std::memcpy(at, Slot(c), Size(c));
    else std::memcpy(Slot(c), at, Size(c));
    last[c % kSlots].store(c, std::memory_order_release);
    copied.fetch_add(1, std::memory_order_release);
    return true;
  }
  void Run(int i) {
    begun[i].store(true);
    at_work.fetch_add(1);
    while (next.load() < n)
      if (!Step()) std::this_thread::yield();
    ended[i].store(true);
  }
};

// A job's threads.  On every way out no chunk is claimed any more and none is being
// copied; threads that have begun are joined, the others are left to `late`.
class ColumnCopy::Crew {
 public:
  Crew(std::shared_ptr<Job> const &job, std::vector<Late> *late) : job_(job), late_(late) {
    for (size_t i = late->size(); i-- > 0;) {
      if (!(*late)[i].job->ended[(*late)[i].index].load()) continue;
      (*late)[i].thread.join();
      late->erase(late->begin() + (long)i);
    }
    wanted_ = (int)std::min<int64_t>(kThreads, job->n);
    if (late->size() >= kThreads) return;  // the processors are taken: no more threads that wait for one
    try {
      late->reserve(late->size() + kThreads);
      threads_.reserve(kThreads);
      for (int i = 0; i < wanted_; ++i) threads_.emplace_back([job, i] { job->Run(i); });
    } catch (std::exception const &) {  // no threads or no memory left: fewer than wished for
    }
  }
  ~Crew() {
    const int64_t claimed = std::min(job_->next.exchange(job_->n), job_->n);
    while (job_->copied.load(std::memory_order_acquire) < claimed) std::this_thread::yield();
    for (int i = 0; i < (int)threads_.size(); ++i) {
      if (job_->begun[i].load()) threads_[i].join();
      else late_->push_back(Late{ std::move(threads_[i]), job_, i });
    }
  }
  // Copies a chunk in the place of a thread that is not at work, or lets others run.
  void Help() {
    if (job_->at_work.load() >= wanted_ || !job_->Step()) std::this_thread::yield();
  }
  bool Short() const { return job_->at_work.load() < wanted_; }

 private:
  std::shared_ptr<Job> job_;
  std::vector<Late> *late_;
  std::vector<std::thread> threads_;
  int wanted_ = 0;
};

void ColumnCopy::Reserve(size_t bytes) {
  if (user_ || bytes < kLeastToHost) return;
  for (auto &e : events_) Check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "column copy event");
  Rings::Get().Enter(bytes);
  user_ = true;
}

ColumnCopy::~ColumnCopy() {
  for (auto &l : late_) l.thread.join();
  GiveBack();
  if (user_) Rings::Get().Leave();
  for (auto &e : events_)
    if (e) (void)hipEventDestroy(e);
}

bool ColumnCopy::Take(size_t bytes, size_t least, hipStream_t stream) {
  if (!user_ || bytes < least) return false;
  Settle();
  ring_ = Rings::Get().Lend(bytes);
  if (ring_) busy_ = stream;
  return ring_ != nullptr;
}

void ColumnCopy::GiveBack() {
  if (ring_) Rings::Get().Return(ring_);
  ring_ = nullptr;
  busy_ = nullptr;
}

void ColumnCopy::Settle() {
  if (busy_) Wait(busy_);
}

void ColumnCopy::Wait(hipStream_t stream) {
  Check(hipStreamSynchronize(stream), "column copy sync");
  if (busy_ == stream) GiveBack();
}

void ColumnCopy::ToHost(void *host, const void *device, size_t bytes, hipStream_t stream) {
  if (!Take(bytes, kLeastToHost, stream)) {
    Check(hipMemcpyAsync(host, device, bytes, hipMemcpyDeviceToHost, stream), "column to host");
    Check(hipStreamSynchronize(stream), "column to host sync");
    return;
  }
  const auto job = std::make_shared<Job>(host, *ring_, bytes, true);
  int64_t issued = 0, filled = 0;
  auto issue = [&] {
    while (issued < job->n && (issued < kSlots || job->Holds(issued - kSlots))) {
      Check(hipMemcpyAsync(job->Slot(issued), static_cast<const char *>(device) + size_t(issued) * job->chunk,
                           job->Size(issued), hipMemcpyDeviceToHost, stream), "column to host");
      Check(hipEventRecord(events_[issued % kSlots], stream), "column to host event");
      ++issued;
    }
  };
  issue();  // the first copies run while the threads start
  {
    Crew crew(job, &late_);
    const int64_t first = std::min<int64_t>(job->n, kSlots);  // till these are filled, threads may still begin
    while (job->copied.load(std::memory_order_acquire) < job->n) {
      if (filled < issued && !(filled >= first && crew.Short() && job->Step())) {
        Check(hipEventSynchronize(events_[filled % kSlots]), "column to host sync");
        job->limit.store(++filled, std::memory_order_release);
      } else if (filled == issued) {  // all slots wait to be emptied, or it is the column's end
        crew.Help();
      }
      issue();
    }
  }
  GiveBack();
}

void ColumnCopy::ToDevice(void *device, const void *host, size_t bytes, hipStream_t stream) {
  if (!Take(bytes, kLeastToDevice, stream)) {
    Check(hipMemcpyAsync(device, host, bytes, hipMemcpyHostToDevice, stream), "column to device");
    return;
  }
  const auto job = std::make_shared<Job>(const_cast<void *>(host), *ring_, bytes, false);
  int64_t drained = 0;
  auto free_slots = [&] { job->limit.store(std::min(job->n, drained + kSlots), std::memory_order_release); };
  free_slots();
  Crew crew(job, &late_);
  for (int64_t c = 0; c < job->n; ++c) {
    // half of the slots on their way to the device, the other half being filled
    for (; c - drained >= kSlots / 2; free_slots()) {
      Check(hipEventSynchronize(events_[drained % kSlots]), "column to device sync");
      ++drained;
    }
    while (!job->Holds(c)) crew.Help();
    Check(hipMemcpyAsync(static_cast<char *>(device) + size_t(c) * job->chunk, job->Slot(c), job->Size(c),
                         hipMemcpyHostToDevice, stream), "column to device");
    Check(hipEventRecord(events_[c % kSlots], stream), "column to device event");
  }
}

}  // namespace mcfd
