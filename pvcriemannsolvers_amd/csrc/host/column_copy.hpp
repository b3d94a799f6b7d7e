// Columns between pageable host memory and the device.
#ifndef MINICFD_HOST_COLUMN_COPY_HPP_
#define MINICFD_HOST_COLUMN_COPY_HPP_

#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

namespace mcfd {

// A column goes through a ring of pinned slots: the stream's copies fill or
// drain the slots while several host threads copy between them and the caller's
// memory.  The caller's side bounds a direct copy: pages that numpy.empty has
// just handed out are zeroed as the copy touches them, by one thread.  The
// threads live for one call, so nothing runs between calls; more than four gain
// nothing.  One copy at a time: callers hold `mutex` over it, over the launches
// that fill or read the same device buffer, and until the stream is drained.
class ColumnCopy {
 public:
  ColumnCopy() = default;
  ColumnCopy(const ColumnCopy &) = delete;
  ColumnCopy &operator=(const ColumnCopy &) = delete;
  ~ColumnCopy();
  // Prepares the ring for columns of up to `bytes`; without it (or where
  // the memory cannot be had) copies are direct.
  void Reserve(size_t bytes);
  // Returns when the column is in `host`.
  void ToHost(void *host, const void *device, size_t bytes, hipStream_t stream);
  // The caller synchronises the stream.
  void ToDevice(void *device, const void *host, size_t bytes, hipStream_t stream);

  std::mutex mutex;

 private:
  static constexpr int kSlots = 16;
  static constexpr int kThreads = 4;
  bool Ring(size_t bytes, size_t least) const;
  static size_t Chunk(size_t bytes);
  // Waits for what may still read or fill the slots: a call that failed leaves its
  // copies in flight, and a copy to the device those that its caller waits for.
  void Settle();
  char *pinned_ = nullptr;
  size_t slot_ = 0;  // bytes of one
  size_t most_ = 0;  // chunks of a column: the slots where the ring is not full, else any number
  hipEvent_t events_[kSlots] = {};
  hipStream_t busy_ = nullptr;  // of those copies
};

}  // namespace mcfd

#endif  // MINICFD_HOST_COLUMN_COPY_HPP_
