// Pools that outlive a call: device scratch, and the pinned blocks that copies
// between a caller's arrays and the device go through. Host code only.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <memory>

namespace ctas {

// Device scratch of a call that waits for its work before it returns. Small
// buffers (up to kScratchBytes) go back to a pool of at most kScratchKept per
// device, since allocating and freeing one costs more than most of the work
// that needs it (about 0.3 ms for the ring filter's column means); any other
// is freed. A buffer is in the hands of one call at a time. done(): the work
// that used it has finished; without it the buffer is freed, which waits.
class Scratch {
 public:
  explicit Scratch(size_t bytes);
  ~Scratch();
  Scratch(const Scratch &) = delete;
  Scratch &operator=(const Scratch &) = delete;
  void *get() const { return p_; }  // null when the allocation failed
  void done() { done_ = true; }

 private:
  void *p_ = nullptr;
  size_t bytes_;
  int dev_ = 0;
  bool done_ = false;
};
constexpr size_t kScratchBytes = size_t{1} << 20;
constexpr int kScratchKept = 4;

// Pinned blocks, events and a stream for copies between a caller's arrays and
// the device. The runtime's own copies of pageable memory move 4 MiB at 15
// GB/s here (33 GB/s at 17 MB, where it pins the caller's pages). With pinned
// blocks the host's copy to or from one runs beside the device's copy of
// another; a kernel makes the latter, since a queued hipMemcpyAsync of a block
// costs tens of microseconds. One slice of 1024 px x 900 angles from and to
// host arrays: 851 us by the runtime, 534 with blocks of 512 KiB, 637 with 1
// MiB, 670 with 256 KiB (643 by hipMemcpyAsync of 1 MiB). Allocating them
// takes milliseconds, so a set goes back to a pool: at most kStagingSets per
// device exist (4 MiB each), one call uses a set at a time, and a call that
// gets none copies as before.
constexpr size_t kStagingBlock = size_t{1} << 19;
constexpr int kStagingBlocks = 8, kStagingSets = 4;
constexpr size_t kStagingMost = size_t{8} << 20;  // larger copies are the runtime's

// Words between a pinned block and device memory, by a kernel on s (capi.hip).
hipError_t staging_copy(void *dst, const void *src, size_t bytes, hipStream_t s);

struct StagingSet;

// A set for one call on device `dev`, given back once nothing of it is in
// flight. None where another device is current: the set's stream and kernel
// would be that device's, and the memory they are given is not (the runtime's
// own copies take any).
class Staging {
 public:
  explicit Staging(int dev);
  ~Staging();
  Staging(const Staging &) = delete;
  Staging &operator=(const Staging &) = delete;

  explicit operator bool() const { return set_ != nullptr; }
  hipEvent_t mark() const;  // an event for the caller's use

  // Queues host -> device copies on s; src may be changed on return.
  hipError_t upload(void *dst, const void *src, size_t bytes, hipStream_t s);
  // Device -> host on the set's stream, complete on return.
  hipError_t download(void *dst, const void *src, size_t bytes);

 private:
  hipError_t wait(int b);  // until block b's last copy of this call is done
  hipError_t copy(int b, void *dst, const void *src, size_t bytes, hipStream_t s);  // with block b

  std::unique_ptr<StagingSet> set_;
  bool busy_[kStagingBlocks] = {};  // block b's event was recorded in this call and not waited for
  int next_ = 0;
};

}  // namespace ctas
