// Ring-artefact filter of sinograms (RingFilter::apply, lct.cpp:295-327):
// subtract from every row the difference between the column mean over
// angles and its box average of half-width `box`. The column
// sums run over the rows in order, and the box sum and the edge
// divisions follow the reference's statement order, so the result matches a
// sequential float implementation bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <string>

#include "ctas_internal.hpp"

namespace ctas {
namespace {

// Column means of ctas_ring_filter_dev_noalloc: a file-scope device array,
// one copy per GPU, held until the process ends. Host code never passes the
// array's name to a kernel (on the host it is a stand-in, not a device
// address): each device's address comes from hipGetSymbolAddress, taken
// once per device with that device current.
constexpr long long kRingScratchFloats = 1LL << 20;  // 4 MiB: S * w <= 1,048,576
__device__ __align__(256) float scratch[kRingScratchFloats];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float *g_scratch_ptr[kMaxDevices] = {};

// Column means. The sum of a column is one chain of additions over the rows
// in order, so a workgroup has 64 columns: its four waves load 64 rows at a
// time into LDS (the next 64 into registers meanwhile) and the first wave
// adds them, a column per lane. Bound by HBM where the columns fill the chip
// (16 x 1800 x 2048: 34 us; one thread per column from memory: 432 us)
// and by the load latency of its N / 64 steps where they do not.
constexpr int kMeanU = 16;  // rows a wave loads per step
__global__ __launch_bounds__(256) void column_mean_kernel(const float *__restrict__ sino, float *__restrict__ avg,
                                                          int N, int w) {
  constexpr int ROWS = 4 * kMeanU;
  __shared__ float tile[2][ROWS][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, s = blockIdx.y;
  const int x = blockIdx.x * 64 + lane, xc = min(x, w - 1);
  const float *p = sino + static_cast<size_t>(s) * N * w + xc;
  float v[kMeanU];
  // rows r0 + wave + 4 j, clamped to the last (those past it are not added)
  auto fetch = [&](int r0) {
#pragma unroll
    for (int j = 0; j < kMeanU; ++j) v[j] = p[static_cast<size_t>(min(r0 + wave + 4 * j, N - 1)) * w];
  };
  auto stage = [&](int b) {
#pragma unroll
    for (int j = 0; j < kMeanU; ++j) tile[b][wave + 4 * j][lane] = v[j];
  };
  fetch(0);
  stage(0);
  float a = 0.0f;
  int b = 0;
  for (int r0 = 0; r0 < N; r0 += ROWS, b ^= 1) {
    __syncthreads();  // tile b is staged, and the sums of tile b ^ 1 are done
    const bool more = r0 + ROWS < N;
    if (more) fetch(r0 + ROWS);
    if (wave == 0) {
      const int m = N - r0;
      if (m >= ROWS) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) a = a + tile[b][r][lane];
      } else {
        for (int r = 0; r < m; ++r) a = a + tile[b][r][lane];
      }
    }
    if (more) stage(b ^ 1);
  }
  if (wave == 0 && x < w) avg[static_cast<size_t>(s) * w + x] = a / static_cast<float>(N);
}

// Row update: block (x, s, z) adds the correction of 256 columns to a chunk
// of rows. Every chunk forms the corrections anew from the means (2 box + 1
// cached reads), so a chunk has at least four times as many rows as that.
// Bound by HBM: 16 x 1800 x 2048 in 77 us (437 us with one chunk).
__global__ __launch_bounds__(256) void ring_apply_kernel(float *__restrict__ sino, const float *__restrict__ avg,
                                                         int N, int w, int box, int chunk) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int s = blockIdx.y;
  if (x >= w) return;
  const float *a = avg + static_cast<size_t>(s) * w;
  float t = 0.0f;
  for (int ii = -box; ii <= box; ++ii) {
    // dstR(w, ii) = [max(0, ii), w-1+min(0, ii)], source x - ii
    const int d0 = ii > 0 ? ii : 0, d1 = w - 1 + (ii < 0 ? ii : 0);
    if (x >= d0 && x <= d1) t = t + a[x - ii];
  }
  if (x >= box && x <= w - 1 - box) t = t / static_cast<float>(2 * box + 1);
  for (int ii = 0; ii < box; ++ii) {
    if (x == ii) t = t / static_cast<float>(box + ii + 1);
    if (x == w - 1 - ii) t = t / static_cast<float>(box + ii + 1);
  }
  t = t - a[x];
  const int r0 = blockIdx.z * chunk, r1 = min(N, r0 + chunk);
  float *p = sino + (static_cast<size_t>(s) * N + r0) * w + x;
#pragma unroll 8
  for (int r = r0; r < r1; ++r, p += w) *p = *p + t;
}

}  // namespace

hipError_t launch_ring(float *d_sino, float *d_avg, int S, int N, int w, int box, hipStream_t s) {
  hipLaunchKernelGGL(column_mean_kernel, dim3((w + 63) / 64, S), dim3(256), 0, s, d_sino, d_avg, N, w);
  const int chunk = static_cast<int>(std::min<long long>(N, std::max(64LL, 4LL * (2LL * box + 1))));
  hipLaunchKernelGGL(ring_apply_kernel, dim3((w + 255) / 256, S, (N + chunk - 1) / chunk), dim3(256), 0, s, d_sino,
                     d_avg, N, w, box, chunk);
  return hipGetLastError();
}

}  // namespace ctas

using namespace ctas;

extern "C" int ctas_ring_filter_dev_noalloc(float *d_sino, int S, int N, int w, int box, void *stream) {
  if (!d_sino || S <= 0 || N <= 0 || w <= 0 || box < 0) return fail(CTAS_E_ARG, "bad arguments");
  if (static_cast<long long>(S) * w > kRingScratchFloats)
    return fail(CTAS_E_ARG, "ring filter without allocation: " + std::to_string(S) + " slices x " +
                                std::to_string(w) + " columns exceed its " + std::to_string(kRingScratchFloats) +
                                " column means of scratch");
  if (box == 0) return CTAS_OK;
  if (int rc = check_ring_box(box, w)) return rc;
  int dev = 0;
  CTAS_HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return fail(CTAS_E_DEVICE, "device index " + std::to_string(dev) + " out of range");
  float *avg = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
      void *p = nullptr;
      CTAS_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
      g_scratch_ptr[dev] = static_cast<float *>(p);
    }
    avg = g_scratch_ptr[dev];
  }
  // column_mean_kernel writes every mean it reads back: nothing to clear
  const hipError_t e = launch_ring(d_sino, avg, S, N, w, box, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return fail(CTAS_E_DEVICE, std::string("ring filter: ") + hipGetErrorString(e));
  return CTAS_OK;
}
