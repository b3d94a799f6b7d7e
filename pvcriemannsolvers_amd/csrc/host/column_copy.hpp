// Columns between pageable host memory and the device.
#ifndef MINICFD_HOST_COLUMN_COPY_HPP_
#define MINICFD_HOST_COLUMN_COPY_HPP_

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace mcfd {

// A column goes through a ring of pinned slots: the stream's copies fill or
// drain the slots while several host threads copy between them and the caller's
// memory.  The caller's side bounds a direct copy: pages that numpy.empty has
// just handed out are zeroed as the copy touches them, by one thread.  The
// threads live for one call and more than four gain nothing.  The caller waits
// for none that has not begun: where the processors are busy (another library's
// threads spinning) that takes milliseconds.  It copies in their place, but only from
// the first ring's end on: till then its own part, the next transfers, comes first
// (48 columns of 0.5 to 10 MB 1 ms a pass slower else).  One
// copy at a time: callers hold `mutex` over it, over the launches that fill or
// read the same device buffer, and until the stream is drained.
//
// The rings belong to the process, as many as there are users, up to four, so that
// pinned memory is bounded and a new handle beside others finds pages that are
// mapped already: a ring's own cost its first copy 0.4 ms per MiB and thread.  The
// last user gives them back.  A new handle's first 4.4 MB to the host, us, with a
// ring per handle / the process's: 770 to 960 / 240 to 280, and on processors that
// another library's threads keep busy 1060 to 6000 / 200 to 330, 1 of 8 at 4000,
// where a thread was stopped at its work (direct 290; a process's first handle 870).
class ColumnCopy {
 public:
  ColumnCopy() = default;
  ColumnCopy(const ColumnCopy &) = delete;
  ColumnCopy &operator=(const ColumnCopy &) = delete;
  ~ColumnCopy();
  // Prepares for columns of up to `bytes`; without it (or where the memory
  // cannot be had, or all rings are lent) copies are direct.
  void Reserve(size_t bytes);
  // Returns when the column is in `host`.
  void ToHost(void *host, const void *device, size_t bytes, hipStream_t stream);
  // The caller waits with Wait().
  void ToDevice(void *device, const void *host, size_t bytes, hipStream_t stream);
  // Waits for the stream.
  void Wait(hipStream_t stream);

  std::mutex mutex;

  struct Ring {  // of kSlots slots at most
    char *pinned;
    size_t bytes;
  };
  static constexpr int kSlots = 16;

 private:
  static constexpr int kThreads = 4;
  struct Job;
  struct Late {  // a thread that had not begun when its call returned
    std::thread thread;
    std::shared_ptr<Job> job;
    int index;
  };
  // A ring for a column of `bytes`, or false for a direct copy.
  bool Take(size_t bytes, size_t least, hipStream_t stream);
  void GiveBack();
  // Waits for what may still read or fill the slots: a call that failed leaves its
  // copies in flight, and a copy to the device those that its caller waits for.
  void Settle();
  class Crew;

  bool user_ = false;  // of the rings
  Ring *ring_ = nullptr;
  hipEvent_t events_[kSlots] = {};
  hipStream_t busy_ = nullptr;  // of the copies in flight
  std::vector<Late> late_;
};

}  // namespace mcfd

#endif  // MINICFD_HOST_COLUMN_COPY_HPP_
