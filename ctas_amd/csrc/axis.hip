// Rotation-axis search (raxis, lct.cpp:1133-1326) with the trial
// reconstructions and their sharpness scores (AverageGradient::apply,
// lct.cpp:872-915) evaluated on the GPU in batches of centres.
//
// Score of one trial slice: the one-sided Gaussian smoothing of
// lct.cpp:837-843 / 878-884 is the circular convolution with
// g[u]*g[v], g[n] = exp(-n^2 / (2 sigma^2)), evaluated separably with the
// taps above 1e-9 (a row pass, then a column pass, both in LDS); then the
// rows [r, w-r) with r = ceil|c| are Sobel-filtered into the matching rows
// of zeroed full-size derivative arrays, and the magnitude is read from the
// top w-2r rows of those arrays (the shape mismatch of lct.cpp:905), the
// border of that block is zeroed and the mean of its positive values is the
// score. The block sums are reduced in a fixed order (deterministic).
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <functional>
#include <memory>
#include <string>
#include <vector>

#include "ctas_internal.hpp"
#include "score_layout.hpp"

namespace ctas {
namespace {

constexpr int kMaxTaps = 64;

struct Taps {
  float g[kMaxTaps];
  int nt;
};

Taps make_taps(float sigma) {
  Taps t{};
  const float sig22 = 2 * sigma * sigma;
  t.nt = 0;
  for (int n = 0; n < kMaxTaps; ++n) {
    const float v = std::exp(-static_cast<float>(n * n) / sig22);
    t.g[n] = v;
    if (v > 1e-9f) t.nt = n + 1;
  }
  return t;
}

// i mod w for i >= -(kMaxTaps + 1); w - 1 past the end, which no valid
// derivative reads.
__device__ __forceinline__ int wrap_index(int i, int w) {
  if (i >= w) return w - 1;
  if (i >= 0) return i;
  i += w;
  return i >= 0 ? i : ((i % w) + w) % w;
}

// dst[k] = sum_n g[n] src[k - n] (n ascending) for the four outputs k = 0..3
// of a line with element stride `st`; src points at output 0.
__device__ __forceinline__ float4 smooth4(const float *src, int st, const Taps &taps) {
  float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f, a3 = 0.0f;
  float x0 = src[0], x1 = src[st], x2 = src[2 * st], x3 = src[3 * st];
#pragma unroll 4
  for (int n = 0; n < taps.nt; ++n) {
    const float g = taps.g[n];
    a0 = a0 + g * x0;
    a1 = a1 + g * x1;
    a2 = a2 + g * x2;
    a3 = a3 + g * x3;
    x3 = x2;
    x2 = x1;
    x1 = x0;
    x0 = src[-min(n + 1, taps.nt - 1) * st];
  }
  return make_float4(a0, a1, a2, a3);
}

// Partial sums of the score of slice k = blockIdx.y over the derivative
// rows and columns of tile blockIdx.x: partial[(k nb + tile) 2 + {0, 1}] =
// {sum of cS, #(cS > 0)}, nb = gridDim.x. The tile of the slice, with the
// rows above and the columns to the left that the one-sided smoothing
// reaches (circularly) and a border of one for the Sobel operator, is read
// into LDS once; smoothing along rows, along columns and the derivatives
// follow there, four outputs per thread in the smoothing so that each LDS read
// serves up to four taps. Bound by LDS reads: nine slices of 2048 px, 8
// taps, 148 us (628 in three passes over memory).
__global__ __launch_bounds__(256) void score_kernel(const float *__restrict__ slices, const float *__restrict__ centres,
                                                    int w, int tiles_x, Taps taps, double *__restrict__ partial) {
  extern __shared__ __align__(16) float score_buf[];
  const ScoreLayout lay = score_layout(taps.nt);
  const int e = lay.reach, rows = lay.rows, cols = lay.cols;
  float *src = score_buf, *mid = score_buf + lay.mid;
  const int tid = threadIdx.x, k = blockIdx.y, nb = gridDim.x;
  const float c = centres[k];
  const int r = static_cast<int>(ceilf(fabsf(c)));
  const int h = w - 2 * r;
  // the full-array row y of lct.cpp:887-912 holds cropped-derivative row
  // y - r (zero above r): rows y = max(1, r) .. h - 2, columns 1 .. w - 2
  const int yy0 = blockIdx.x / tiles_x * kScoreTH, x0 = 1 + blockIdx.x % tiles_x * kScoreTW;
  const int yy_lo = r < 1 ? 1 - r : 0, yy_hi = h - 2 - r;
  double sm = 0.0, cnt = 0.0;
  if (yy0 <= yy_hi) {
    const float *sl = slices + static_cast<size_t>(k) * w * w;
    // slice rows r + yy0 - 1 - e .., columns x0 - 1 - e ..
    for (int b = tid & 63; b < cols; b += 64) {
      const float *column = sl + wrap_index(x0 - 1 - e + b, w);
      for (int a0 = tid >> 6; a0 < rows; a0 += 32) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = column[static_cast<size_t>(wrap_index(r + yy0 - 1 - e + a0 + 4 * j, w)) * w];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (a0 + 4 * j < rows) src[(a0 + 4 * j) * cols + b] = v[j];
      }
    }
    __syncthreads();
    if (taps.nt > 0) {
      for (int i = tid; i < rows * (kScoreSW / 4); i += 256) {
        const int a = i / (kScoreSW / 4), b = 4 * (i - a * (kScoreSW / 4));
        *reinterpret_cast<float4 *>(mid + a * kScoreSW + b) = smooth4(src + a * cols + e + b, 1, taps);
      }
      __syncthreads();
      for (int i = tid; i < (kScoreSH / 4) * kScoreSW; i += 256) {
        const int a = 4 * (i / kScoreSW), b = i % kScoreSW;
        const float4 v = smooth4(mid + (e + a) * kScoreSW + b, kScoreSW, taps);
        float *d = src + a * kScoreSW + b;
        d[0] = v.x;
        d[kScoreSW] = v.y;
        d[2 * kScoreSW] = v.z;
        d[3 * kScoreSW] = v.w;
      }
      __syncthreads();
    }
    // rows above the cropped slice count as zero (those below are not reached)
    auto at = [&](int yy, int x) {
      return yy < 0 ? 0.0f : src[(yy - yy0 + 1) * kScoreSW + (x - x0 + 1)];
    };
    const int x = x0 + (tid & 63);
    for (int j = tid >> 6; j < kScoreTH; j += 4) {
      const int yy = yy0 + j;
      if (yy < yy_lo || yy > yy_hi || x > w - 2) continue;
      // the statement order of lct.cpp:887-902
      const float a = at(yy - 1, x - 1), b = at(yy - 1, x), d = at(yy - 1, x + 1);
      const float p = at(yy, x - 1), q = at(yy, x + 1);
      const float u = at(yy + 1, x - 1), v = at(yy + 1, x), z = at(yy + 1, x + 1);
      float dH = 0.0f, dV = 0.0f;
      dH = dH + -1.0f * z;
      dH = dH + -2.0f * v;
      dH = dH + -1.0f * u;
      dH = dH + 1.0f * d;
      dH = dH + 2.0f * b;
      dH = dH + 1.0f * a;
      dV = dV + -1.0f * z;
      dV = dV + -2.0f * q;
      dV = dV + -1.0f * d;
      dV = dV + 1.0f * u;
      dV = dV + 2.0f * p;
      dV = dV + 1.0f * a;
      const float m = sqrtf(dH * dH + dV * dV);
      sm += m;
      // #(cS > 0) of lct.cpp:912: the reference's float-FFT smoothing leaves
      // round-off in every pixel, so then every derivative pixel counts.
      cnt += (taps.nt > 0 || m > 0.0f) ? 1.0 : 0.0;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    sm += __shfl_xor(sm, o);
    cnt += __shfl_xor(cnt, o);
  }
  __shared__ double ps[4], pc[4];
  if ((tid & 63) == 0) {
    ps[tid >> 6] = sm;
    pc[tid >> 6] = cnt;
  }
  __syncthreads();
  if (tid == 0) {
    double *out = partial + (static_cast<size_t>(k) * nb + blockIdx.x) * 2;
    out[0] = (ps[0] + ps[1]) + (ps[2] + ps[3]);
    out[1] = (pc[0] + pc[1]) + (pc[2] + pc[3]);
  }
}

// Score of slice k (blockIdx.x): the nb partials summed in a fixed order.
__global__ __launch_bounds__(256) void score_finish_kernel(const double *__restrict__ partial,
                                                           float *__restrict__ scores, int nb) {
  const int k = blockIdx.x;
  double s = 0.0, c = 0.0;
  for (int b = threadIdx.x; b < nb; b += blockDim.x) {
    s += partial[(static_cast<size_t>(k) * nb + b) * 2];
    c += partial[(static_cast<size_t>(k) * nb + b) * 2 + 1];
  }
  __shared__ double ps[256], pc[256];
  ps[threadIdx.x] = s;
  pc[threadIdx.x] = c;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) {
      ps[threadIdx.x] += ps[threadIdx.x + o];
      pc[threadIdx.x] += pc[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const float sm = static_cast<float>(ps[0]);
    scores[k] = pc[0] > 0.0 ? sm / static_cast<float>(pc[0]) : 0.0f;
  }
}

}  // namespace

int score_tiles(int w) {
  return ((w + kScoreTW - 1) / kScoreTW) * ((w + kScoreTH - 1) / kScoreTH);
}

hipError_t launch_ag_scores(const float *d_slices, int n, int w, const float *d_centres, float sigma,
                            double *d_partial, float *d_scores, hipStream_t s) {
  Taps taps{};
  if (sigma > 1.0f) taps = make_taps(sigma);
  const int nb = score_tiles(w);
  hipLaunchKernelGGL(score_kernel, dim3(nb, n), dim3(256), sizeof(float) * score_layout(taps.nt).floats, s, d_slices, d_centres, w,
                     (w + kScoreTW - 1) / kScoreTW, taps, d_partial);
  if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  hipLaunchKernelGGL(score_finish_kernel, dim3(n), dim3(256), 0, s, d_partial, d_scores, nb);
  return hipGetLastError();
}

namespace {

template <typename T>
int grow_buf(T *&ptr, size_t &cap, size_t bytes) {
  if (bytes <= cap && ptr) return CTAS_OK;
  if (ptr) (void)hipFree(ptr);
  ptr = nullptr;
  cap = 0;
  void *p = nullptr;
  if (hipMalloc(&p, std::max<size_t>(bytes, 256)) != hipSuccess)
    return fail(CTAS_E_NOMEM, "device allocation of " + std::to_string(bytes) + " bytes failed");
  ptr = static_cast<T *>(p);
  cap = bytes;
  return CTAS_OK;
}


}  // namespace

// improveMe (lct.cpp:1108-1129): bisection towards the lower neighbour.
// The bracket around offsets[at] is halved on its wider side until both
// sides are within eps; a probe that scores no better than the current best
// becomes that side's edge, a better one the new best (the old best then
// closes the other side).
float improve_me(float eps, const std::vector<float> &offsets, const std::vector<float> &scores, int at, int dir,
                 const std::function<float(float)> &score_at, int *rc) {
  float left = offsets[at - dir];
  float right = offsets[at + dir];
  float best = offsets[at];
  float best_score = scores[at];
  while (std::fabs(left - best) > eps || std::fabs(best - right) > eps) {
    const bool left_wider = std::fabs(left - best) > std::fabs(best - right);
    float &wide = left_wider ? left : right;
    float &narrow = left_wider ? right : left;
    const float probe = (best + wide) / 2;
    const float probe_score = score_at(probe);
    if (*rc) return best;
    if (best_score <= probe_score) {
      wide = probe;
    } else {
      best_score = probe_score;
      narrow = best;
      best = probe;
    }
  }
  return best;
}

namespace {

struct HandleGuard {
  ctas_fbp *h = nullptr;
  ~HandleGuard() {
    if (h) ctas_fbp_destroy(h);
  }
};

}  // namespace
}  // namespace ctas

using namespace ctas;

extern "C" int ctas_axis_scores(ctas_fbp *h, const float *axisR, int n, float *scores) {
  if (!h || !axisR || !scores || n <= 0) return fail(CTAS_E_ARG, "bad arguments");
  if (h->kept_slices < 1) return fail(CTAS_E_STATE, "no filtered sinogram on the device: call ctas_fbp_sino first");
  const int w = h->w;
  const float sigma = static_cast<float>(step_rad(h->anarc, h->N) * static_cast<float>(w) / M_PI);
  const size_t ww = static_cast<size_t>(w) * w;
  for (int k0 = 0; k0 < n; k0 += kScoreChunk) {
    const int m = std::min(kScoreChunk, n - k0);
    std::vector<float> centres(m);
    for (int i = 0; i < m; ++i)
      centres[i] = static_cast<float>(static_cast<double>(axisR[k0 + i]) - 0.5 * (w - 1));
    if (int rc = grow_buf(h->d_out, h->out_cap, sizeof(float) * ww * m)) return rc;
    if (int rc = grow_buf(h->d_partial, h->score_cap, sizeof(double) * 2 * score_tiles(w) * m)) return rc;
    if (!h->d_centres) {
      if (hipMalloc(&h->d_centres, sizeof(float) * kScoreChunk) != hipSuccess ||
          hipMalloc(&h->d_scores, sizeof(float) * kScoreChunk) != hipSuccess)
        return fail(CTAS_E_NOMEM, "allocation failed");
    }
    // all on the handle's stream: the centres' upload, the trial slices, the
    // scores and their download, then one wait (centres outlives it)
    CTAS_HIP_TRY(hipMemcpyAsync(h->d_centres, centres.data(), sizeof(float) * m, hipMemcpyHostToDevice, h->stream));
    if (int rc = ctas_fbp_repeat_dev(h, 0, h->d_out, centres.data(), m, h->stream)) return rc;
    CTAS_HIP_TRY(launch_ag_scores(h->d_out, m, w, h->d_centres, sigma, h->d_partial, h->d_scores, h->stream));
    CTAS_HIP_TRY(hipMemcpyAsync(scores + k0, h->d_scores, sizeof(float) * m, hipMemcpyDeviceToHost, h->stream));
    CTAS_HIP_TRY(hipStreamSynchronize(h->stream));
  }
  return CTAS_OK;
}

namespace ctas {
namespace {

// ---- 0/180-degree registration (raxis(proj0, proj180, maxDev)) ----------
// Column profile sum_r |p0 - 1| + |p180 - 1| (double terms added to a float
// per column, rows in order, lct.cpp:1226-1235). The sums are serial chains,
// so a column is a lane, and one wave per workgroup spreads the columns over
// the CUs; the rows of a chain are loaded 16 at a time. Bound by the chain:
// 2048 rows of 2048 columns take 104 us (7.3 ms, the serial sums below
// included, in one workgroup; those now take 38 us).
__global__ __launch_bounds__(64) void pair_profile_kernel(const float *__restrict__ p0,
                                                          const float *__restrict__ p180, int rows, int w,
                                                          float *__restrict__ prof) {
  const int x = blockIdx.x * 64 + threadIdx.x;
  if (x >= w) return;
  float acc = 0.0f;
  auto add = [&](float a, float b) {
    acc = static_cast<float>(acc + (fabs(static_cast<double>(a) - 1.0) + fabs(static_cast<double>(b) - 1.0)));
  };
  constexpr int U = 16;
  int r = 0;
  for (; r + U <= rows; r += U) {
    float a[U], b[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const size_t i = static_cast<size_t>(r + j) * w + x;
      a[j] = p0[i];
      b[j] = p180[i];
    }
#pragma unroll
    for (int j = 0; j < U; ++j) add(a[j], b[j]);
  }
  for (; r < rows; ++r) {
    const size_t i = static_cast<size_t>(r) * w + x;
    add(p0[i], p180[i]);
  }
  prof[x] = acc;
}

// The serial sums of lct.cpp:1236-1251, each a workgroup whose first lane
// adds what all lanes stage: block 0 the profile's sum and moment (out[0],
// out[1]), blocks 1 and 2 the edge columns of the mirrored p180 (its first
// column is p180's last and vice versa; out[2], out[3]).
__global__ __launch_bounds__(256) void pair_sums_kernel(const float *__restrict__ prof,
                                                        const float *__restrict__ p180, int rows, int w,
                                                        double *__restrict__ out) {
  constexpr int C = 1024;
  __shared__ float stage[C];
  const int what = blockIdx.x, n = what == 0 ? w : rows;
  double sum = 0.0, moment = 0.0;
  for (int i0 = 0; i0 < n; i0 += C) {
    const int m = min(C, n - i0);
    __syncthreads();
    for (int i = threadIdx.x; i < m; i += 256)
      stage[i] = what == 0 ? prof[i0 + i] : p180[static_cast<size_t>(i0 + i) * w + (what == 1 ? w - 1 : 0)];
    __syncthreads();
    if (threadIdx.x != 0) continue;
    if (what == 0) {
#pragma unroll 8
      for (int i = 0; i < m; ++i) {
        sum += stage[i];
        moment += static_cast<double>(static_cast<float>(i0 + i) * stage[i]);
      }
    } else {
#pragma unroll 8
      for (int i = 0; i < m; ++i) sum += stage[i];
    }
  }
  if (threadIdx.x != 0) return;
  if (what == 0) {
    out[0] = sum;
    out[1] = moment;
  } else {
    out[1 + what] = sum;
  }
}

// Registration errors of k trial shifts (calcErr of lct.cpp:1255-1270): sum
// over rows and columns of (p180r(col - sh) - p0)^2, p180r the mirrored p180,
// `aver` outside the overlap, each square in float and summed in double.
// Block (b, c) takes R rows and eight trials: the rows of p180 lie mirrored
// in LDS, each sample of p0 is loaded once for the eight trials, and the
// lanes' sums are reduced in a fixed order. part[t][b] receives the block's
// sum of trial t. Bound by the conversions and double additions: the 65
// trials of a sweep over 2048 x 2048 samples and the 33 of a bracket take
// 77 us each on average; one workgroup per trial, reading both projections
// from memory, took 8 ms for the sweep and as much for each probe of the
// bisection.
constexpr int kPairTrials = 8;
__global__ __launch_bounds__(256) void pair_err_kernel(const float *__restrict__ p0, const float *__restrict__ p180,
                                                       int rows, int w, int R, const int *__restrict__ shifts, int k,
                                                       float aver, double *__restrict__ part) {
  extern __shared__ float mirrored[];  // [R][w]
  const int tid = threadIdx.x, r0 = blockIdx.x * R, nr = min(R, rows - r0), t0 = blockIdx.y * kPairTrials;
  for (int r = 0; r < nr; ++r)
    for (int x = tid; x < w; x += 256) mirrored[r * w + (w - 1 - x)] = p180[static_cast<size_t>(r0 + r) * w + x];
  int sh[kPairTrials];
  double acc[kPairTrials];
#pragma unroll
  for (int t = 0; t < kPairTrials; ++t) {
    sh[t] = shifts[min(t0 + t, k - 1)];
    acc[t] = 0.0;
  }
  __syncthreads();
  for (int r = 0; r < nr; ++r) {
    const float *line = mirrored + r * w;
    const float *ref = p0 + static_cast<size_t>(r0 + r) * w;
    for (int col = tid; col < w; col += 256) {
      const float v = ref[col];
#pragma unroll
      for (int t = 0; t < kPairTrials; ++t) {
        const int src = col - sh[t];
        const bool in = static_cast<unsigned>(src) < static_cast<unsigned>(w);
        const float s = line[in ? src : 0];
        const float d = (in ? s : aver) - v;
        acc[t] += static_cast<double>(d * d);
      }
    }
  }
  __shared__ double wave_sum[4][kPairTrials];
#pragma unroll
  for (int t = 0; t < kPairTrials; ++t) {
    double a = acc[t];
    for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o);
    if ((tid & 63) == 0) wave_sum[tid >> 6][t] = a;
  }
  __syncthreads();
  if (tid < kPairTrials && t0 + tid < k)
    part[static_cast<size_t>(t0 + tid) * gridDim.x + blockIdx.x] =
        (wave_sum[0][tid] + wave_sum[1][tid]) + (wave_sum[2][tid] + wave_sum[3][tid]);
}

// Sum of trial blockIdx.x over the nb row blocks, in a fixed order.
__global__ __launch_bounds__(256) void pair_err_sum_kernel(const double *__restrict__ part, int nb,
                                                           double *__restrict__ out) {
  __shared__ double red[256];
  const double *p = part + static_cast<size_t>(blockIdx.x) * nb;
  double acc = 0.0;
  for (int i = threadIdx.x; i < nb; i += 256) acc += p[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (static_cast<int>(threadIdx.x) < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = red[0];
}

}  // namespace
}  // namespace ctas

using namespace ctas;

// raxis(proj0, proj180, maxDev) (lct.cpp:1217-1294): registration of the
// 0 and 180 degree projections. The profile and the error sums of every
// trial shift run on the GPU; the sweep and the bisection are host logic.
extern "C" int ctas_raxis_pair(const float *p0, const float *p180, int rows, int w, float maxDev, float *result) {
  if (!p0 || !p180 || !result) return fail(CTAS_E_ARG, "null argument");
  if (maxDev < 0 || maxDev > 0.5f)
    return fail(CTAS_E_ARG, "Invalid maximum relative shift of the rotation axis " + std::to_string(maxDev) +
                                ". Must be within [0, 0.5] range.");
  if (rows <= 0 || w <= 0) return fail(CTAS_E_ARG, "Empty input projections.");
  if (w > 16384) return fail(CTAS_E_ARG, "projection width above 16384");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(CTAS_E_DEVICE, "no HIP device is available");
  const float mid = static_cast<float>(0.5 * (w - 1));
  const size_t n = static_cast<size_t>(rows) * w;
  const int kStep = 16;
  const int n_trials = static_cast<int>(1 + 2 * (maxDev == 0.0f ? 1.0f : maxDev * static_cast<float>(w) / kStep));
  // device: p0, p180, profile results, trial shifts, their sums
  // the trial shifts of one evaluation: the sweep, a chunk of the walk, or the
  // whole shifts of the bisection's bracket (2 kStep + 1 and a margin)
  constexpr int kWalkChunk = 16;
  const int max_trials = std::max(n_trials, 2 * kStep + 8);
  // rows per workgroup: four where that leaves 256 of them, and within 64 KiB
  // of LDS
  const int R = std::max(1, std::min({4, rows / 256, 16384 / w}));
  const int nb = (rows + R - 1) / R;
  struct Buf {
    void *p = nullptr;
    ~Buf() {
      if (p) (void)hipFree(p);
    }
  } buf;
  auto up = [](size_t b) { return (b + 255) & ~static_cast<size_t>(255); };
  const size_t off_prof = up(2 * n * sizeof(float)), off_sum = off_prof + up(sizeof(float) * w),
               off_sh = off_sum + 256, off_acc = off_sh + up(sizeof(int) * max_trials),
               off_part = off_acc + up(sizeof(double) * max_trials);
  if (hipMalloc(&buf.p, off_part + sizeof(double) * max_trials * static_cast<size_t>(nb)) != hipSuccess)
    return fail(CTAS_E_NOMEM, "device allocation failed");
  char *base = static_cast<char *>(buf.p);
  float *d_p0 = reinterpret_cast<float *>(base), *d_p180 = d_p0 + n;
  float *d_prof = reinterpret_cast<float *>(base + off_prof);
  double *d_sum = reinterpret_cast<double *>(base + off_sum), *d_acc = reinterpret_cast<double *>(base + off_acc),
         *d_part = reinterpret_cast<double *>(base + off_part);
  int *d_sh = reinterpret_cast<int *>(base + off_sh);
  CTAS_HIP_TRY(hipMemcpy(d_p0, p0, n * sizeof(float), hipMemcpyHostToDevice));
  CTAS_HIP_TRY(hipMemcpy(d_p180, p180, n * sizeof(float), hipMemcpyHostToDevice));
  hipLaunchKernelGGL(pair_profile_kernel, dim3((w + 63) / 64), dim3(64), 0, nullptr, d_p0, d_p180, rows, w, d_prof);
  hipLaunchKernelGGL(pair_sums_kernel, dim3(3), dim3(256), 0, nullptr, d_prof, d_p180, rows, w, d_sum);
  CTAS_HIP_TRY(hipGetLastError());
  double sums[4];
  CTAS_HIP_TRY(hipMemcpy(sums, d_sum, sizeof sums, hipMemcpyDeviceToHost));
  if (sums[0] == 0.0) return fail(CTAS_E_AXIS, "Impossible input projection averaging to zero.");
  const float seed = static_cast<float>(sums[1]) / static_cast<float>(sums[0]);
  const float mean_level = (static_cast<float>(sums[2]) + static_cast<float>(sums[3])) / static_cast<float>(2 * rows);
  int dev_rc = CTAS_OK;
  // errors of the whole shifts sh[0..k)
  auto whole_errs = [&](const std::vector<int> &sh, float *e) {
    const int k = static_cast<int>(sh.size());
    if (dev_rc != CTAS_OK) return;
    if (k < 1 || k > max_trials) {  // what the device buffers hold
      dev_rc = fail(CTAS_E_AXIS, "Failed to calculate rotation centre.");
      return;
    }
    std::vector<double> acc(k);
    if (hipMemcpy(d_sh, sh.data(), sizeof(int) * k, hipMemcpyHostToDevice) != hipSuccess) {
      dev_rc = fail(CTAS_E_DEVICE, "registration: upload failed");
      return;
    }
    hipLaunchKernelGGL(pair_err_kernel, dim3(nb, (k + kPairTrials - 1) / kPairTrials), dim3(256),
                       sizeof(float) * R * w, nullptr, d_p0, d_p180, rows, w, R, d_sh, k, mean_level, d_part);
    hipLaunchKernelGGL(pair_err_sum_kernel, dim3(k), dim3(256), 0, nullptr, d_part, nb, d_acc);
    if (hipGetLastError() != hipSuccess ||
        hipMemcpy(acc.data(), d_acc, sizeof(double) * k, hipMemcpyDeviceToHost) != hipSuccess) {
      dev_rc = fail(CTAS_E_DEVICE, "registration: error sums failed on the device");
      return;
    }
    for (int i = 0; i < k; ++i) e[i] = std::sqrt(static_cast<float>(acc[i]));
  };
  // a trial's error depends on its offset truncated to whole pixels
  auto errs = [&](const float *xs, int k, float *e) {
    std::vector<int> sh(k);
    for (int i = 0; i < k; ++i) sh[i] = static_cast<int>(static_cast<long>(xs[i]));
    whole_errs(sh, e);
  };
  // improveMe within the bracket [lo, hi]: its probes take at most
  // 2 kStep + 1 whole shifts, evaluated together beforehand
  auto refine = [&](const std::vector<float> &at, const std::vector<float> &e, int idx, int dir, int *rc) -> float {
    const float a = at[idx - dir], b = at[idx + dir];
    const int lo = static_cast<int>(static_cast<long>(std::min(a, b))), hi = static_cast<int>(static_cast<long>(std::max(a, b)));
    std::vector<int> sh(hi - lo + 1);
    for (size_t i = 0; i < sh.size(); ++i) sh[i] = lo + static_cast<int>(i);
    std::vector<float> err(sh.size());
    whole_errs(sh, err.data());
    if (dev_rc != CTAS_OK) return 0.0f;
    return improve_me(1.0f, at, e, idx, dir, [&](float x) { return err[static_cast<int>(static_cast<long>(x)) - lo]; }, rc);
  };
  std::vector<float> offsets(n_trials), errors(n_trials);
  for (int ii = 0; ii < n_trials; ++ii) offsets[ii] = 2 * (seed - mid) + static_cast<float>(kStep * (ii - (n_trials - 1) / 2));
  errs(offsets.data(), n_trials, errors.data());
  if (dev_rc != CTAS_OK) return dev_rc;
  int idx = -1;
  float best_error = FLT_MAX;
  for (int i = 1; i < n_trials - 1; ++i)
    if (errors[i] < errors[i - 1] && errors[i] < errors[i + 1] && errors[i] < best_error) best_error = errors[idx = i];
  int rc = CTAS_OK;
  if (idx >= 0) {
    *result = mid + 0.5f * refine(offsets, errors, idx, 1, &rc);
    return dev_rc != CTAS_OK ? dev_rc : rc;
  }
  idx = errors[0] < errors[n_trials - 1] ? 0 : n_trials - 1;
  const int dir = idx == 0 ? -1 : 1;
  best_error = errors[idx];
  const int walk_limit = static_cast<int>((static_cast<float>(w / 2) - static_cast<float>(dir) * offsets[idx]) / kStep);
  if (walk_limit <= 0) return fail(CTAS_E_AXIS, "Failed to calculate rotation centre.");
  std::vector<float> walk_offsets(walk_limit + 2), walk_errors(walk_limit + 2);
  // a sweep of one trial (maxDev w < 8) has no neighbour: the next grid point
  // is the bracket's other side
  walk_offsets[0] = n_trials > 1 ? offsets[idx - dir] : offsets[idx] - static_cast<float>(dir * kStep);
  walk_offsets[1] = offsets[idx];
  walk_errors[1] = errors[idx];
  int walk_best = 1;
  for (int i = 0; i < walk_limit; ++i) walk_offsets[i + 2] = offsets[idx] + static_cast<float>(dir * (i + 1) * kStep);
  for (int i = 0; i < walk_limit; ++i) {
    if (i % kWalkChunk == 0) {
      errs(walk_offsets.data() + i + 2, std::min(kWalkChunk, walk_limit - i), walk_errors.data() + i + 2);
      if (dev_rc != CTAS_OK) return dev_rc;
    }
    if (walk_errors[i + 2] < best_error) {
      best_error = walk_errors[i + 2];
      walk_best = i + 2;
    } else {
      break;
    }
  }
  if (walk_best == walk_limit + 1) return fail(CTAS_E_AXIS, "Failed to calculate rotation centre.");
  *result = mid + 0.5f * refine(walk_offsets, walk_errors, walk_best, dir, &rc);
  return dev_rc != CTAS_OK ? dev_rc : rc;
}

// raxis(sino, anarc, maxDev, algo) (lct.cpp:1133-1212). The trial
// reconstructions of the sweep run as one batch; the directional walk is
// evaluated in batches and cut at its first non-improving trial, which is
// the sequential order of AGinThread::exexafter2 (lct.cpp:1028-1040); the
// bisection is sequential.
extern "C" int ctas_raxis(const float *sino, int N, int w, float anarc, float maxDev, int algo, float *result) {
  if (!sino || !result) return fail(CTAS_E_ARG, "null argument");
  if (N < 3 || w < 3)
    return fail(CTAS_E_AXIS, "Shape of input sinogram (" + std::to_string(N) + "," + std::to_string(w) +
                                 ") is less than minimal (3,3).");
  const float arc = arc_rad(anarc, N);
  if (arc == 0.0f) return fail(CTAS_E_AXIS, "Zero sinogram arc.");
  if (std::fabs(arc) < static_cast<float>(M_PI))
    return fail(CTAS_E_AXIS, "Sinogram arc " + std::to_string(std::fabs(arc) * 180 / M_PI) + " is less than 180 degree.");
  const float kShiftLimit = 0.25f;
  if (maxDev < 0 || maxDev > kShiftLimit)
    return fail(CTAS_E_AXIS, "Invalid maximum relative shift of the rotation axis " + std::to_string(maxDev) + ".");
  const float mid = static_cast<float>(0.5 * (w - 1));
  float seed = 0.0f;
  if (algo == 0 || algo == 2) {
    const int half_turn = static_cast<int>((N - 1) * M_PI / std::fabs(arc_rad(anarc, N)));
    const int n_rows = N - half_turn;
    if (n_rows <= 0) return fail(CTAS_E_AXIS, "No opposite projections in the sinogram.");
    std::vector<float> r0(static_cast<size_t>(n_rows) * w), r180(static_cast<size_t>(n_rows) * w);
    for (int j = 0; j < n_rows; ++j)
      for (int x = 0; x < w; ++x) {
        r0[static_cast<size_t>(j) * w + x] = sino[static_cast<size_t>(j) * w + x] + 1;
        r180[static_cast<size_t>(j) * w + x] = sino[static_cast<size_t>(j + half_turn) * w + x] + 1;
      }
    float q = 0.0f;
    if (int rc = ctas_raxis_pair(r0.data(), r180.data(), n_rows, w, std::min(maxDev, 0.5f), &q)) return rc;
    if (algo == 0) {
      *result = q;
      return CTAS_OK;
    }
    seed = q;
  } else if (algo == 1) {
    seed = mid;
  } else if (algo == 3) {
    std::vector<float> profile(w, 0.0f);
    for (int j = 0; j < N; ++j)
      for (int x = 0; x < w; ++x) profile[x] = profile[x] + sino[static_cast<size_t>(j) * w + x];
    const float mx = *std::max_element(profile.begin(), profile.end());
    const float mn = *std::min_element(profile.begin(), profile.end());
    // lct.cpp:1168-1180 only ends its scans at a sample above the
    // threshold; a constant projection has none.
    if (!(mx > mn)) return fail(CTAS_E_AXIS, "Constant projection: no edge above the threshold.");
    const float threshold = static_cast<float>(0.1 * mx + 0.9 * mn);
    int a = 0, b = w - 1;
    while (!(profile[a] > threshold)) ++a;
    while (!(profile[b] > threshold)) --b;
    seed = (static_cast<float>(a) + static_cast<float>(b)) / 2.0f;
  } else {
    return fail(CTAS_E_AXIS, "Unknown algorithm for rotation axis " + std::to_string(algo) + ".");
  }
  if (std::fabs(seed - mid) / w > maxDev)
    return fail(CTAS_E_AXIS, "Rotation axis relative shift " + std::to_string(std::fabs(seed - mid) / w) +
                                 " is larger than maximum shift " + std::to_string(maxDev) + ".");
  const float box_fraction = static_cast<float>(1.0 - 2.0 * (maxDev + std::fabs(seed - mid) / w));
  if (box_fraction < 0.5f)
    return fail(CTAS_E_AXIS, "Relative box size " + std::to_string(box_fraction) + " is less than miminum window of 0.5.");

  // AverageGradient (lct.cpp:818-844): ABS contrast, RAMP, the sinogram
  // filtered once.
  HandleGuard g;
  if (int rc = ctas_fbp_create(&g.h, w, N, CTAS_CONTRAST_ABS, CTAS_FILTER_RAMP, 0.0f, anarc, 0)) return rc;
  std::vector<float> copy(sino, sino + static_cast<size_t>(N) * w);
  if (int rc = ctas_fbp_sino(g.h, copy.data())) return rc;
  int rc = CTAS_OK;
  auto score_at = [&](float x) -> float {
    float axes = mid + x, s = 0.0f;
    if (!rc) rc = ctas_axis_scores(g.h, &axes, 1, &s);
    return s;
  };

  const int kStep = 8;
  const int n_trials = static_cast<int>(1 + 2 * (maxDev == 0.0f ? 1.0f : maxDev * static_cast<float>(w) / kStep));
  const int half = (n_trials - 1) / 2;
  const float seed_offset = seed - mid;
  std::vector<float> offsets(n_trials), scores(n_trials), axes(n_trials);
  for (int k = 0; k < n_trials; ++k) {
    offsets[k] = seed_offset + static_cast<float>(kStep * (k - half));
    axes[k] = mid + offsets[k];
  }
  if ((rc = ctas_axis_scores(g.h, axes.data(), n_trials, scores.data()))) return rc;
  int best_at = 0;
  float best_score = FLT_MAX;
  for (int i = 1; i < n_trials - 1; ++i)
    if (scores[i] < scores[i - 1] && scores[i] < scores[i + 1] && scores[i] < best_score) {
      best_at = i;
      best_score = scores[i];
    }
  int dir = 1;
  if (!best_at) {
    const int idx = scores[0] < scores[n_trials - 1] ? 0 : n_trials - 1;
    dir = idx == 0 ? -1 : 1;
    // two grid points back; beyond the sweep where that has one or two trials
    const int walk_from = static_cast<int>(seed_offset + static_cast<float>(kStep * (idx - dir * 2 - half)));
    const int walk_limit = static_cast<int>(static_cast<float>(w) * kShiftLimit - static_cast<float>(dir * walk_from / kStep));
    if (walk_limit <= 0) return fail(CTAS_E_AXIS, "Impossible number of n_trials.");
    std::vector<float> walk_offsets, walk_scores;
    bool stop = false;
    constexpr int kWalkChunk = 8;
    for (int k0 = 0; k0 < walk_limit && !stop; k0 += kWalkChunk) {
      const int m = std::min(kWalkChunk, walk_limit - k0);
      std::vector<float> a(m), s(m);
      for (int i = 0; i < m; ++i) a[i] = mid + (static_cast<float>(walk_from) + static_cast<float>(kStep * (k0 + i) * dir));
      if ((rc = ctas_axis_scores(g.h, a.data(), m, s.data()))) return rc;
      for (int i = 0; i < m && !stop; ++i) {
        walk_offsets.push_back(static_cast<float>(walk_from) + static_cast<float>(kStep * (k0 + i) * dir));
        walk_scores.push_back(s[i]);
        if (s[i] < best_score) {
          best_score = s[i];
          best_at = k0 + i;
        } else {
          stop = true;
        }
      }
    }
    if (best_at == walk_limit - 1 || best_at == 0) {
      *result = seed;
      return CTAS_OK;
    }
    offsets = walk_offsets;
    scores = walk_scores;
  }
  const float rf = improve_me(0.25f, offsets, scores, best_at, dir, score_at, &rc);
  if (rc) return rc;
  *result = mid + rf;
  return CTAS_OK;
}
