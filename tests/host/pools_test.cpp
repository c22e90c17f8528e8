// The pools of pools.cpp on a host-only stand-in for HIP; `pools_test <case>`
// exits with 0 when the case holds.
#include "pools.hpp"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <set>
#include <string>
#include <vector>

namespace {
int g_device = 0;       // the current one
int g_calls = 0;        // every HIP call
bool g_refuse = false;  // allocations fail
std::set<hipStream_t> g_streams;                  // those that exist
std::map<hipEvent_t, hipStream_t> g_recorded;     // the stream of an event's last record
hipError_t g_last = hipSuccess;

hipError_t call(hipError_t e = hipSuccess) {
  ++g_calls;
  if (e != hipSuccess) g_last = e;
  return e;
}
hipError_t allocate(void **p, size_t bytes) {
  if (g_refuse) return call(hipErrorOutOfMemory);
  *p = std::aligned_alloc(256, (bytes + 255) / 256 * 256);
  return call();
}
void check(bool ok, const char *what) {
  if (ok) return;
  std::printf("failed: %s\n", what);
  std::exit(1);
}
}  // namespace

hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
hipError_t hipGetDevice(int *dev) {
  *dev = g_device;
  return call();
}
hipError_t hipMalloc(void **p, size_t bytes) { return allocate(p, bytes); }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { return allocate(p, bytes); }
hipError_t hipFree(void *p) {
  std::free(p);
  return call();
}
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipMemcpy(void *dst, const void *src, size_t bytes, hipMemcpyKind) {
  std::memcpy(dst, src, bytes);
  return call();
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return allocate(reinterpret_cast<void **>(e), 1); }
hipError_t hipEventDestroy(hipEvent_t e) { return hipFree(e); }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  g_recorded[e] = s;
  return call();
}
// An event may be waited for while the stream that it was recorded on is there.
hipError_t hipEventSynchronize(hipEvent_t e) {
  const auto at = g_recorded.find(e);
  if (at != g_recorded.end() && at->second && !g_streams.count(at->second)) return call(hipErrorInvalidValue);
  return call();
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  const hipError_t e = allocate(reinterpret_cast<void **>(s), 1);
  if (e == hipSuccess) g_streams.insert(*s);
  return e;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  g_streams.erase(s);
  return hipFree(s);
}
hipError_t hipStreamSynchronize(hipStream_t) { return call(); }

namespace ctas {
hipError_t staging_copy(void *dst, const void *src, size_t bytes, hipStream_t) {
  std::memcpy(dst, src, bytes);
  call();
  return hipGetLastError();  // as after a launch
}
}  // namespace ctas

using namespace ctas;

// Copies of every number of blocks arrive whole.
void copies() {
  for (size_t n : {size_t{1}, size_t{33}, kStagingBlock / 4, kStagingBlock / 4 + 1, kStagingBlock * 2 + 3,
                   kStagingMost / 4, kStagingMost / 4 + 1}) {
    std::vector<float> a(n), dev(n), b(n, -1.0f);
    for (size_t i = 0; i < n; ++i) a[i] = static_cast<float>(i % 1000);
    Staging st(0);
    check(static_cast<bool>(st), "a set for the current device");
    check(st.upload(dev.data(), a.data(), 4 * n, nullptr) == hipSuccess, "upload");
    check(st.download(b.data(), dev.data(), 4 * n) == hipSuccess, "download");
    check(a == b, "what comes back");
  }
}

// A call whose device is not the current one gets no set, and one that has one
// takes none from the others.
void device() {
  g_device = 1;
  check(!Staging(0), "no set for device 0 while device 1 is current");
  std::vector<std::unique_ptr<Staging>> held;
  for (int k = 0; k < kStagingSets + 1; ++k) held.emplace_back(new Staging(1));
  for (int k = 0; k < kStagingSets; ++k) check(static_cast<bool>(*held[k]), "a set for each call");
  check(!*held[kStagingSets], "as many sets as the limit");
  g_device = 0;
  check(static_cast<bool>(Staging(0)), "the other device's sets are its own");
}

// A set goes from a handle to the next after the first one's stream is gone.
void streams() {
  std::vector<float> a(kStagingMost / 4), dev(a.size()), b(a.size());
  for (int handle = 0; handle < 3; ++handle) {
    for (size_t i = 0; i < a.size(); ++i) a[i] = static_cast<float>((i + handle) % 1000);
    hipStream_t s = nullptr;
    check(hipStreamCreateWithFlags(&s, hipStreamNonBlocking) == hipSuccess, "a stream");
    {
      Staging st(0);
      check(st.upload(dev.data(), a.data(), 4 * a.size(), s) == hipSuccess, "upload");
      check(st.download(b.data(), dev.data(), handle ? 4 : 4 * a.size()) == hipSuccess, "download");
    }
    check(hipGetLastError() == hipSuccess, "no wait for a record on a stream that is gone");
    (void)hipStreamDestroy(s);
  }
}

// Without memory a call goes on without a set or scratch, and the failed
// allocation is not what its next launch reports. Afterwards all is as before.
void refused() {
  float a = 1.0f, b = 0.0f;
  g_refuse = true;
  check(!Staging(0), "no set");
  check(staging_copy(&b, &a, sizeof a, nullptr) == hipSuccess, "the launch after a refused set");
  check(Scratch(100).get() == nullptr && Scratch(2 * kScratchBytes).get() == nullptr, "no scratch");
  check(staging_copy(&b, &a, sizeof a, nullptr) == hipSuccess, "the launch after refused scratch");
  g_refuse = false;
  device();
  copies();
}

// The calls made when main ended; what runs after the static objects'
// destructors holds the count against it.
int g_at_end = -1;
__attribute__((destructor)) void after_main() {
  if (g_at_end < 0 || g_calls == g_at_end) return;
  std::printf("failed: %d HIP calls after the end of main\n", g_calls - g_at_end);
  std::fflush(stdout);
  std::_Exit(1);
}

// The pools' destructors leave the runtime alone.
void end() {
  copies();
  { Scratch a(100); a.done(); }
  g_at_end = g_calls;
}

int main(int argc, char **argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "copies") copies();
  else if (what == "device") device();
  else if (what == "streams") streams();
  else if (what == "refused") refused();
  else if (what == "end") end();
  else return 2;
  return 0;
}
