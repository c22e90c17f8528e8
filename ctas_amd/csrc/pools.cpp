// Pools that outlive a call (pools.hpp).
#include "pools.hpp"

#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

namespace ctas {

namespace {
// Whether an allocation succeeded. The error of one that failed would be
// reported by the next launch that asks hipGetLastError, and what follows does
// without the memory.
bool allocated(hipError_t e) {
  if (e == hipSuccess) return true;
  (void)hipGetLastError();
  return false;
}

std::mutex g_scratch_pool_mu;
std::map<int, std::vector<void *>> g_scratch_pool;  // by device, kScratchBytes each
}  // namespace

Scratch::Scratch(size_t bytes) : bytes_(std::max<size_t>(bytes, 1)) {
  if (hipGetDevice(&dev_) != hipSuccess) return;
  if (bytes_ <= kScratchBytes) {
    bytes_ = kScratchBytes;
    std::lock_guard<std::mutex> lk(g_scratch_pool_mu);
    auto &pool = g_scratch_pool[dev_];
    if (!pool.empty()) {
      p_ = pool.back();
      pool.pop_back();
      return;
    }
  }
  if (!allocated(hipMalloc(&p_, bytes_))) p_ = nullptr;
}

Scratch::~Scratch() {
  if (!p_) return;
  if (done_ && bytes_ == kScratchBytes) {
    std::lock_guard<std::mutex> lk(g_scratch_pool_mu);
    auto &pool = g_scratch_pool[dev_];
    if (pool.size() < static_cast<size_t>(kScratchKept)) {
      pool.push_back(p_);
      return;
    }
  }
  (void)hipFree(p_);
}

struct StagingSet {
  int dev = 0;
  unsigned char *block[kStagingBlocks] = {};
  hipEvent_t free[kStagingBlocks] = {};  // the last copy that used the block
  hipEvent_t mark = nullptr;
  hipStream_t stream = nullptr;

  ~StagingSet() {
    if (stream) (void)hipStreamDestroy(stream);
    if (mark) (void)hipEventDestroy(mark);
    for (hipEvent_t e : free)
      if (e) (void)hipEventDestroy(e);
    if (block[0]) (void)hipHostFree(block[0]);
  }
  bool make() {
    if (hipGetDevice(&dev) != hipSuccess ||
        !allocated(hipHostMalloc(reinterpret_cast<void **>(&block[0]), kStagingBlock * kStagingBlocks)))
      return false;
    for (int b = 0; b < kStagingBlocks; ++b) {
      block[b] = block[0] + kStagingBlock * b;
      if (!allocated(hipEventCreateWithFlags(&free[b], hipEventDisableTiming))) return false;
    }
    return allocated(hipEventCreateWithFlags(&mark, hipEventDisableTiming)) &&
           allocated(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
  }
};

namespace {
std::mutex g_staging_mu;
struct DeviceSets {
  StagingSet *idle[kStagingSets];  // the sets not in use
  int n_idle = 0, made = 0;
};
// Raw pointers: the sets end with the process, since the runtime may be gone
// before this file's static objects are.
std::map<int, DeviceSets> g_staging;
}  // namespace

Staging::Staging(int dev) {
  int current = -1;
  if (hipGetDevice(&current) != hipSuccess || current != dev) return;
  {
    std::lock_guard<std::mutex> lk(g_staging_mu);
    DeviceSets &d = g_staging[dev];
    if (d.n_idle > 0) {
      set_.reset(d.idle[--d.n_idle]);
      return;
    }
    if (d.made >= kStagingSets) return;
    ++d.made;
  }
  set_.reset(new StagingSet);
  if (set_->make()) return;
  set_.reset();
  std::lock_guard<std::mutex> lk(g_staging_mu);
  --g_staging[dev].made;
}

Staging::~Staging() {
  if (!set_) return;
  (void)hipStreamSynchronize(set_->stream);
  for (int b = 0; b < kStagingBlocks; ++b) (void)wait(b);
  std::lock_guard<std::mutex> lk(g_staging_mu);
  DeviceSets &d = g_staging[set_->dev];
  d.idle[d.n_idle++] = set_.release();  // no more than were made
}

hipEvent_t Staging::mark() const { return set_->mark; }

// A set outlives the streams of the handles that it served, and the runtime
// looks at the stream that an event was last recorded on. So a call waits for
// its own records only, while its stream is there; the set comes to it idle.
hipError_t Staging::wait(int b) {
  if (!busy_[b]) return hipSuccess;
  busy_[b] = false;
  return hipEventSynchronize(set_->free[b]);
}

hipError_t Staging::copy(int b, void *dst, const void *src, size_t bytes, hipStream_t s) {
  if (hipError_t e = staging_copy(dst, src, bytes, s); e != hipSuccess) return e;
  const hipError_t e = hipEventRecord(set_->free[b], s);
  busy_[b] = e == hipSuccess;
  return e;
}

hipError_t Staging::upload(void *dst, const void *src, size_t bytes, hipStream_t s) {
  if (bytes > kStagingMost) return hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice);
  for (size_t off = 0; off < bytes; off += kStagingBlock, next_ = (next_ + 1) % kStagingBlocks) {
    const size_t n = std::min(kStagingBlock, bytes - off);
    const int b = next_;
    if (hipError_t e = wait(b); e != hipSuccess) return e;
    std::memcpy(set_->block[b], static_cast<const unsigned char *>(src) + off, n);
    if (hipError_t e = copy(b, static_cast<unsigned char *>(dst) + off, set_->block[b], n, s); e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t Staging::download(void *dst, const void *src, size_t bytes) {
  if (bytes > kStagingMost) {
    if (hipError_t e = hipStreamSynchronize(set_->stream); e != hipSuccess) return e;
    return hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
  }
  const size_t chunks = (bytes + kStagingBlock - 1) / kStagingBlock;
  auto size = [&](size_t c) { return std::min(kStagingBlock, bytes - c * kStagingBlock); };
  auto queue = [&](size_t c) -> hipError_t {
    const int b = static_cast<int>(c % kStagingBlocks);
    if (hipError_t e = wait(b); e != hipSuccess) return e;
    return copy(b, set_->block[b], static_cast<const unsigned char *>(src) + c * kStagingBlock, size(c), set_->stream);
  };
  for (size_t c = 0; c < std::min<size_t>(chunks, kStagingBlocks); ++c)
    if (hipError_t e = queue(c); e != hipSuccess) return e;
  for (size_t c = 0; c < chunks; ++c) {
    const int b = static_cast<int>(c % kStagingBlocks);
    if (hipError_t e = wait(b); e != hipSuccess) return e;
    std::memcpy(static_cast<unsigned char *>(dst) + c * kStagingBlock, set_->block[b], size(c));
    if (c + kStagingBlocks < chunks)
      if (hipError_t e = queue(c + kStagingBlocks); e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace ctas
