// Learned front end of the rotation-axis search: a small BF16 CNN that
// predicts the centre offset, and a confidence, from a sinogram downsampled
// to 180 angles x 256 detector bins plus its copy turned by 180 degrees.
//
// Network (245,554 parameters): four 3x3 convolutions (2->32, 32->32, 32->64,
// 64->64, padding 1, leaky ReLU (slope 1/64), 2x2 max pooling after each) on
// 2x180x256, then a 11264->16 fully connected layer with leaky ReLU and a
// 16->2 output (offset in
// downsampled detector bins, confidence logit). Activations and weights are
// bfloat16; every product of the convolutions and of the first fully connected
// layer runs on the matrix cores (v_mfma_f32_16x16x32_bf16, float32
// accumulation), sums that are split over workgroups reduced in a fixed order:
// * conv_kernel: a convolution forward, with its pooling, or (the stencil
//   mirrored, the weights transposed) the gradient of its input, from a patch
//   of the input in LDS;
// * wgrad_kernel, and wgrad_taps_kernel for the first layer: the weight
//   gradients, split over the pixels;
// * gemm_kernel, whose operands small functors gather: the first fully
//   connected layer, forward and backward.
// head_kernel ends the forward pass, loss_kernel begins the backward one.
// Training is Adam on float32 master weights; the bfloat16 copies feed the next
// step.
//
// Training data are made by the engine: seeded ellipse phantoms (plus small
// dense inclusions) projected analytically on the GPU with photon noise,
// then reduced to the network's input on the GPU.
//
// Searches that use the network:
// * ctas_axis_find: the sweep of trial centres on a fixed grid (the
//   AverageGradient score of lct.cpp:872-915 at every grid offset, argmin)
//   is narrowed to a window around the network's estimate that grows until
//   its lowest score is interior; below the confidence threshold the whole
//   grid is swept. Without a network it is the plain sweep.
// * ctas_raxis_cnn: raxis algorithm 1 (lct.cpp:1133-1212) with its 8-px
//   sweep replaced by the estimate and improveMe (lct.cpp:1108-1129) run
//   from the bracket +-4 px around it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <fstream>
#include <memory>
#include <optional>
#include <random>
#include <string>
#include <vector>

#include "ctas_internal.hpp"
#include "pools.hpp"

namespace ctas {
namespace cnn {

typedef float f4 __attribute__((ext_vector_type(4)));

// to nearest even, one conversion instruction (bits by hand take seven)
__device__ __forceinline__ uint16_t bf16_rne(float v) {
  return __builtin_bit_cast(uint16_t, static_cast<__bf16>(v));
}
__device__ __forceinline__ float bf16_f(uint16_t h) { return __uint_as_float(static_cast<uint32_t>(h) << 16); }

constexpr int kFeatA = 180, kFeatW = 256;  // feature map: angles x detector bins
// Slope of the leaky ReLU on the negative side (a power of two, so scaled
// gradients round like the unscaled ones).
constexpr float kLeak = 0.015625f;

__device__ __forceinline__ float leaky(float v) { return v > 0.0f ? v : kLeak * v; }
constexpr int kBT = 64;                    // GEMM block tile (M and N)

// ---- generic GEMM: C[m][n] = sum_k A(m, k) B(k, n) -------------------------
// Block: 256 threads = 4 waves, 64x64 C tile, each wave 32x32 as 2x2 tiles
// of gfx950's v_mfma_f32_16x16x32_bf16. K advances by 32 through LDS. Operand
// layout of that instruction: lane l holds A[l%16][8(l/16)+j] and
// B[8(l/16)+j][l%16] (j = 0..7, eight bf16 in four registers); the result
// D[4(l/16)+r][l%16] (r = 0..3). Both tiles sit in LDS with K contiguous
// ([row][k] for A, [col][k] for B, rows padded to 40 elements), so that a
// lane's eight operands are one 16-byte read; the operand functors gather
// eight consecutive k of one row or column per thread, written as one
// 16-byte store.
// gridDim.z splits K into ranges of k_chunk; each split writes its own
// partial (the store functor gets the split index).
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
constexpr int kKS = 32, kKP = kKS + 8;  // K per step, padded LDS row

template <class FA, class FB, class FC>
__global__ __launch_bounds__(256) void gemm_kernel(FA fa, FB fb, FC fc, int M, int N, int K, int k_chunk) {
  __shared__ __align__(16) uint16_t As[kBT][kKP];
  __shared__ __align__(16) uint16_t Bs[kBT][kKP];
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * kBT, n0 = blockIdx.x * kBT;
  const int kb = blockIdx.z * k_chunk, ke = min(K, kb + k_chunk);
  const int wave = tid >> 6, lane = tid & 63;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const int si = tid >> 2, sk = (tid & 3) * 8;  // staging: row / column si, k offset sk
  f4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = kb; k0 < ke; k0 += kKS) {
    u16x8 va, vb;
    const int m = m0 + si, n = n0 + si;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = k0 + sk + j;
      va[j] = (m < M && k < ke) ? fa(m, k) : static_cast<uint16_t>(0);
      vb[j] = (n < N && k < ke) ? fb(k, n) : static_cast<uint16_t>(0);
    }
    *reinterpret_cast<u16x8 *>(&As[si][sk]) = va;
    *reinterpret_cast<u16x8 *>(&Bs[si][sk]) = vb;
    __syncthreads();
    const int r16 = lane & 15, k8 = (lane >> 4) * 8;
    bf16x8 a[2], b[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      a[t] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u16x8 *>(&As[wm + 16 * t + r16][k8]));
      b[t] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u16x8 *>(&Bs[wn + 16 * t + r16][k8]));
    }
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
      for (int ni = 0; ni < 2; ++ni)
        acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[mi], b[ni], acc[mi][ni], 0, 0, 0);
    __syncthreads();
  }
  const int col = lane & 15, row4 = (lane >> 4) * 4;
#pragma unroll
  for (int mi = 0; mi < 2; ++mi)
#pragma unroll
    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + 16 * mi + row4 + r, n = n0 + wn + 16 * ni + col;
        if (m < M && n < N) fc(m, n, acc[mi][ni][r], blockIdx.z);
      }
}

template <class FA, class FB, class FC>
hipError_t gemm(FA fa, FB fb, FC fc, int M, int N, int K, hipStream_t s, int splits = 1) {
  int chunk = (K + splits - 1) / splits;
  chunk = (chunk + kKS - 1) & ~(kKS - 1);
  splits = (K + chunk - 1) / chunk;
  const dim3 grid((N + kBT - 1) / kBT, (M + kBT - 1) / kBT, splits);
  hipLaunchKernelGGL((gemm_kernel<FA, FB, FC>), grid, dim3(256), 0, s, fa, fb, fc, M, N, K, chunk);
  return hipGetLastError();
}

// ---- the network -----------------------------------------------------------------
struct Layer {
  int cin, cout, H, W;  // conv: input channels, output channels, spatial size
};
constexpr Layer kConv[4] = {{2, 32, 180, 256}, {32, 32, 90, 128}, {32, 64, 45, 64}, {64, 64, 22, 32}};
constexpr int kF = 64 * 11 * 16, kH1 = 16, kOut = 2;

// ---- operand functors ---------------------------------------------------------
struct DenseA {  // A[m][k] bf16, row stride ld
  const uint16_t *p;
  int ld;
  __device__ uint16_t operator()(int m, int k) const { return p[static_cast<size_t>(m) * ld + k]; }
};
struct DenseAT {  // A(m, k) = P[k][m] bf16 (transposed), row stride ld
  const uint16_t *p;
  int ld;
  __device__ uint16_t operator()(int m, int k) const { return p[static_cast<size_t>(k) * ld + m]; }
};
// gradient of the pre-activation: g = d(post) * (post > 0 ? 1 : kLeak), as bf16
__device__ __forceinline__ uint16_t relu_grad(const float *d, const uint16_t *post, size_t i) {
  return bf16_rne(bf16_f(post[i]) > 0.0f ? d[i] : kLeak * d[i]);
}
struct GradFlatA {  // A(o, b) = g[b][o] (fp32 gradient, ReLU-masked by post when given)
  const float *d;
  const uint16_t *post;
  int O;
  __device__ uint16_t operator()(int o, int b) const {
    const size_t i = static_cast<size_t>(b) * O + o;
    return post ? relu_grad(d, post, i) : bf16_rne(d[i]);
  }
};
struct GradFlatB {  // B(o, b) = g[b][o]
  GradFlatA f;
  __device__ uint16_t operator()(int o, int b) const { return f(o, b); }
};
struct ActB {  // B(k, n) = act[n][k] (flattened activations per sample)
  const uint16_t *p;
  int F;
  __device__ uint16_t operator()(int k, int n) const { return p[static_cast<size_t>(n) * F + k]; }
};
struct ActBT {  // B(n, k) = act[n][k]
  const uint16_t *p;
  int F;
  __device__ uint16_t operator()(int n, int k) const { return p[static_cast<size_t>(n) * F + k]; }
};

// ---- store functors -------------------------------------------------------------
struct StoreDX {  // dx[b][ci][y][x] (fp32)
  float *dx;
  int C, H, W;
  __device__ void operator()(int ci, int n, float v, int) const {
    const int hw = H * W, b = n / hw, p = n - b * hw;
    dx[(static_cast<size_t>(b) * C + ci) * hw + p] = v;
  }
};
struct StorePartial {  // ws[split][m][n]
  float *ws;
  int M, N;
  __device__ void operator()(int m, int n, float v, int z) const {
    ws[(static_cast<size_t>(z) * M + m) * N + n] = v;
  }
};
struct StoreFlatDX {  // dx[b][f] fp32 from C(f, b)
  float *dx;
  int F;
  __device__ void operator()(int f, int b, float v, int) const { dx[static_cast<size_t>(b) * F + f] = v; }
};

// ---- elementwise kernels -------------------------------------------------------------
// What the backward pass has to know of a window of the pooling: its first
// maximum's place (two bits: row, column) and whether that is positive.
__device__ __forceinline__ uint32_t pool_code(uint16_t a, uint16_t b, uint16_t c, uint16_t d) {
  const float v[4] = {bf16_f(a), bf16_f(b), bf16_f(c), bf16_f(d)};
  uint32_t at = 0;
  float best = v[0];
#pragma unroll
  for (int k = 1; k < 4; ++k)
    if (v[k] > best) {
      best = v[k];
      at = k;
    }
  return at | (best > 0.0f ? 4u : 0u);
}

// Backward of the pooling and of the leaky ReLU, and the bias gradient, in
// one pass over a channel of a sample (block (co, b)): the pooled gradient dy
// goes to the first maximum of its window, scaled by the slope of that
// post-activation, as bf16 (the operand of the products that follow; every
// other pixel gets zero, rows beyond the pooled extent too); part[b][co]
// receives its sum before rounding. A thread takes four windows: one read of
// their codes, one of dy, two writes. Bound by HBM, whose bytes are the
// writes and half as many reads. Layers two to four (the first forms its
// gradient in wgrad_taps_kernel): 14, 9 and 6 us for 64 samples (10 a layer on
// average; 158 with the gradient in float32 and its bias sums apart, the first
// layer's among them).
__global__ __launch_bounds__(256) void pool_bwd(const uint8_t *__restrict__ code, const float *__restrict__ dy,
                                                uint16_t *__restrict__ g, float *__restrict__ part, int C, int H,
                                                int W) {
  const int co = blockIdx.x, b = blockIdx.y;
  const int Ho = H / 2, Wo = W / 2, Q = Wo / 4;  // W is a multiple of 8
  const size_t plane = static_cast<size_t>(b) * C + co;
  uint16_t *gp = g + plane * H * W;
  const float4 *d4 = reinterpret_cast<const float4 *>(dy + plane * Ho * Wo);
  const uint32_t *c4 = reinterpret_cast<const uint32_t *>(code + plane * Ho * Wo);
  float s = 0.0f;
  for (int i = threadIdx.x; i < Ho * Q; i += 256) {
    const int yo = i / Q, q = i - yo * Q;
    const size_t at = static_cast<size_t>(2 * yo) * W + 8 * q;
    const uint32_t c = c4[i];
    const float4 d = d4[i];
    const float dv[4] = {d.x, d.y, d.z, d.w};
    u16x8 g0, g1;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float gv = c & (4u << (8 * j)) ? dv[j] : kLeak * dv[j];
      s += gv;
      const uint32_t am = c >> (8 * j) & 3u;
      const uint16_t h = bf16_rne(gv);
      g0[2 * j] = am == 0 ? h : 0;
      g0[2 * j + 1] = am == 1 ? h : 0;
      g1[2 * j] = am == 2 ? h : 0;
      g1[2 * j + 1] = am == 3 ? h : 0;
    }
    *reinterpret_cast<u16x8 *>(gp + at) = g0;
    *reinterpret_cast<u16x8 *>(gp + at + W) = g1;
  }
  for (int i = 2 * Ho * (W / 8) + threadIdx.x; i < H * (W / 8); i += 256)
    *reinterpret_cast<u16x8 *>(gp + static_cast<size_t>(8) * i) = u16x8{};
  __shared__ float red[256];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[static_cast<size_t>(b) * C + co] = red[0];
}

// Weight gradient of a convolution, split over the pixels: ws[z][co][c] =
// sum over the pixels of split z of g[co][pixel] x[ci][pixel + tap], c = ci*9
// + tap, 32 pixels per matrix instruction in pixel order. Both operands of
// the instruction are eight consecutive pixels of one row per lane, and
// neighbouring lanes take 16 rows: loaded so, a load touches 64 pieces of
// memory and not 16, and the L1 binds. A wave therefore loads its rows of 32
// pixels as they lie, the next steps' while the current one is multiplied, and
// takes its operands from LDS, which also gives the pixels beside an octet for
// the horizontal taps. It takes all output channels and all nine taps of 16
// input channels. Four waves of a workgroup take a quarter of its pixels each
// and add their sums through LDS: a wave per SIMD with a quarter of the splits
// to write and to reduce, whatever the layer's size. Bound by the latency of a
// step. 64 samples, layers two to four: 43, 21 and 14 us (51, 21 and 15 with
// operands loaded by their lanes; 55, 33 and 26 so with a split per wave, 704 to
// 44 of them; 380 on average through the general product).
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// octet d moved one pixel right (lo: the pixel before it in the upper half)
// or left (hi: the pixel after it in the lower half)
__device__ __forceinline__ u32x4 octet_right(u32x4 d, uint32_t lo) {
  return u32x4{(d.x << 16) | (lo >> 16), (d.y << 16) | (d.x >> 16), (d.z << 16) | (d.y >> 16), (d.w << 16) | (d.z >> 16)};
}
__device__ __forceinline__ u32x4 octet_left(u32x4 d, uint32_t hi) {
  return u32x4{(d.x >> 16) | (d.y << 16), (d.y >> 16) | (d.z << 16), (d.z >> 16) | (d.w << 16), (d.w >> 16) | (hi << 16)};
}

template <int CIN, int COUT, int H, int W>
__global__ __launch_bounds__(256, 2) void wgrad_kernel(const uint16_t *__restrict__ g, const uint16_t *__restrict__ x,
                                                   float *__restrict__ ws, int K, int chunk) {
  constexpr int N = CIN * 9, MT = COUT / 16, HW = H * W;
  static_assert(W % 32 == 0 && CIN % 16 == 0, "32 pixels of one row and 16 channels per step");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r16 = lane & 15, g8 = (lane >> 4) * 8;
  const int z = blockIdx.x;
  const int kb = __builtin_amdgcn_readfirstlane(z * chunk + wave * (chunk / 4)), ke = min(K, kb + chunk / 4);
  // A wave's operands in LDS: rows of 32 pixels, g's of 16*MT channels, and x's
  // of three lines and 16 channels with a pair of pixels on either side
  // (elements 6 and 40); pitches whose 16 rows fall into different banks.
  constexpr int PA = 40, PB = 56, STAGE = MT * 16 * PA + 48 * PB;
  constexpr int RS = 16 * 9 + 4;  // padded row of the sums: 16 input channels and their taps
  __shared__ __align__(16) uint16_t lds[4 * (STAGE > 2 * 16 * RS ? STAGE : 2 * 16 * RS)];
  uint16_t *sa = lds + wave * STAGE, *sb = sa + MT * 16 * PA;
  const int lr = lane >> 2, lo = 8 * (lane & 3);                        // the octet a lane loads: row, column
  const int ed = lane >> 5, eside = lane >> 4 & 1, eat = eside ? 40 : 6;  // its pairs: line ed and line 2 of channel r16
  constexpr int U = MT > 2 ? 2 : 4;  // steps of loads in flight
  struct Step {
    u32x4 a[MT], b[3];
    uint32_t edge[2];
    uint32_t row[3], beside, live;  // masks of what lies inside the image and the split
  } st[U];
  // Branch-free, and masked when used: a branch would wait for its loads.
  auto load = [&](int pn, Step &s) {
    const bool live = pn < ke;
    const int p = live ? pn : ke - 32;  // past the end the last step again, masked
    const int b = p / HW, q = p - b * HW, y = q / W, x0 = q - y * W;  // uniform
    const uint16_t *ga = g + static_cast<size_t>(b) * COUT * HW + q;
#pragma unroll
    for (int m = 0; m < MT; ++m) s.a[m] = *reinterpret_cast<const u32x4 *>(ga + (16 * m + lr) * HW + lo);
    const uint16_t *xb = x + (static_cast<size_t>(b) * CIN + blockIdx.y * 16) * HW + x0;
    int line[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int yy = y + d - 1;
      const bool row = yy >= 0 && yy < H;
      line[d] = (row ? yy : y) * W;
      s.b[d] = *reinterpret_cast<const u32x4 *>(xb + lr * HW + line[d] + lo);
      s.row[d] = row && live ? ~0u : 0u;
    }
    const int left = x0 > 0 ? -2 : 0, right = x0 < W - 32 ? 32 : 0, beside = eside ? right : left;
    s.edge[0] = *reinterpret_cast<const uint32_t *>(xb + r16 * HW + (ed ? line[1] : line[0]) + beside);
    s.edge[1] = *reinterpret_cast<const uint32_t *>(xb + r16 * HW + line[2] + beside);
    s.beside = beside ? ~0u : 0u;
    s.live = live ? ~0u : 0u;
  };
  f4 acc[MT][9];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < 9; ++t) acc[m][t] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < U; ++u) load(kb + 32 * u, st[u]);
  for (int p0 = kb; p0 < ke; p0 += 32 * U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = p0 + 32 * u;
#pragma unroll
      for (int m = 0; m < MT; ++m) *reinterpret_cast<u32x4 *>(sa + (16 * m + lr) * PA + lo) = st[u].a[m] & st[u].live;
#pragma unroll
      for (int d = 0; d < 3; ++d)
        *reinterpret_cast<u32x4 *>(sb + (16 * d + lr) * PB + 8 + lo) = st[u].b[d] & st[u].row[d];
      *reinterpret_cast<uint32_t *>(sb + (16 * ed + r16) * PB + eat) =
          st[u].edge[0] & (st[u].beside & (ed ? st[u].row[1] : st[u].row[0]));
      if (ed == 0) *reinterpret_cast<uint32_t *>(sb + (32 + r16) * PB + eat) = st[u].edge[1] & (st[u].beside & st[u].row[2]);
      // one wave: its LDS operations are in order, only the compiler's are not
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      bf16x8 a[MT], bb[9];
#pragma unroll
      for (int m = 0; m < MT; ++m) a[m] = *reinterpret_cast<const bf16x8 *>(sa + (16 * m + r16) * PA + g8);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const uint16_t *at = sb + (16 * d + r16) * PB + 8 + g8;
        const u32x4 o = *reinterpret_cast<const u32x4 *>(at);
        bb[3 * d] = __builtin_bit_cast(bf16x8, octet_right(o, *reinterpret_cast<const uint32_t *>(at - 2)));
        bb[3 * d + 1] = __builtin_bit_cast(bf16x8, o);
        bb[3 * d + 2] = __builtin_bit_cast(bf16x8, octet_left(o, *reinterpret_cast<const uint32_t *>(at + 8)));
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < 9; ++t) acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], bb[t], acc[m][t], 0, 0, 0);
      // the next step's operands are not waited for before these products
      __builtin_amdgcn_sched_barrier(0);
      // two steps are one 128-byte line of each row: loaded together
      if (u & 1) {
        load(p + 32 * (U - 1), st[u - 1]);
        load(p + 32 * U, st[u]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  // the four waves' sums, 16 output channels at a time
  float *part = reinterpret_cast<float *>(lds);
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) part[(wave * 16 + (lane >> 4) * 4 + r) * RS + r16 * 9 + t] = acc[m][t][r];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      const int i = threadIdx.x + 256 * j, co = i / 144, c = i - co * 144, at = co * RS + c;
      ws[(static_cast<size_t>(z) * COUT + 16 * m + co) * N + blockIdx.y * 144 + c] =
          ((part[at] + part[16 * RS + at]) + part[32 * RS + at]) + part[48 * RS + at];
    }
  }
}

// The same for the network's two-channel input, which has no gradient of its
// own: nothing else reads the gradient of the layer's pre-activation, so it is
// formed here, from the pooled gradient dy and the windows' codes, a pair of
// rows at a time, and never stored; ws[z][COUT*18 + co] receives its sum before
// rounding (bias). The input's 18 columns (channel and tap) are two tiles of
// lanes; a step's octets of it are loaded once, one per lane, with the image's
// border as zeros, and each lane takes those of its own taps from LDS (read
// from memory at a pixel's shift they bound the kernel: 66 us). K counts steps
// of two rows' 32 pixels. Bound by the latency of a step with two in flight
// (four: 48 us). 64 samples: 45 us, where pooling backward and the product took
// 51 and 79 and wrote and read 190 MB between them.
typedef uint16_t u16x8u __attribute__((ext_vector_type(8), aligned(2)));
template <int CIN, int COUT, int H, int W>
__global__ __launch_bounds__(64, 2) void wgrad_taps_kernel(const uint8_t *__restrict__ code, const float *__restrict__ dy,
                                                        const uint16_t *__restrict__ x, float *__restrict__ ws, int K,
                                                        int chunk) {
  constexpr int N = CIN * 9, MT = COUT / 16, NT = (N + 15) / 16, HW = H * W, PW = W / 2, PHW = HW / 4;
  constexpr int SR = 4 * CIN, SW = 48, OCT = SW / 8;  // rows and columns of a step's input: its border and octets
  static_assert(W % 32 == 0 && H % 2 == 0, "32 pixels of two rows of one window row per step");
  static_assert(SR * OCT <= 64, "one octet of the input per lane");
  __shared__ __align__(16) uint16_t rows[2][SR * SW];
  const int lane = threadIdx.x, r16 = lane & 15, g8 = (lane >> 4) * 8;
  const int z = blockIdx.x, kb = z * chunk, ke = min(K, kb + chunk);
  int at0[NT], edge[NT], dxc[NT];  // the lane's octet in `rows`, the pair beside it, its shift
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int c = t * 16 + r16, cc = c < N ? c : 0, ci = cc / 9, r = cc - 9 * ci;
    dxc[t] = r % 3 - 1;
    at0[t] = (4 * ci + r / 3) * SW + 8 + g8;
    edge[t] = at0[t] + (dxc[t] < 0 ? -2 : 8);
  }
  const int sr = min(lane / OCT, SR - 1), sci = sr >> 2, sy = (sr & 3) - 1, sx = 8 * (lane % OCT) - 8;  // staged octet
  constexpr int U = 2;  // steps of loads in flight
  struct Step {
    float4 d[MT];
    uint32_t c[MT];
    u32x4 x;
    uint32_t in;
  } st[U];
  auto load = [&](int pn, Step &s) {  // step p: 32 columns of window row yo of sample b
    const int p = min(pn, ke - 1);    // past the end the last step again, masked
    const int i = 32 * p, b = i / (H / 2 * W), q = i - b * (H / 2 * W), yo = q / W, x0 = q - yo * W;  // uniform
    const size_t at = static_cast<size_t>(b) * COUT * PHW + yo * PW + x0 / 2;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int o = (16 * m + r16) * PHW + g8 / 2;
      s.d[m] = *reinterpret_cast<const float4 *>(dy + at + o);
      s.c[m] = *reinterpret_cast<const uint32_t *>(code + at + o);
    }
    const int yy = 2 * yo + sy, xx = x0 + sx;
    const bool in = yy >= 0 && yy < H && xx >= 0 && xx < W;
    // the caller's input is aligned to its elements only
    s.x = __builtin_bit_cast(u32x4, *reinterpret_cast<const u16x8u *>(
                                        x + static_cast<size_t>(b) * CIN * HW + (in ? sci * HW + yy * W + xx : 0)));
    s.in = in && pn < ke ? ~0u : 0u;
  };
  f4 acc[MT][NT];
  float bias[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    bias[m] = 0.0f;
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[m][t] = f4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int u = 0; u < U; ++u) load(kb + u, st[u]);
  for (int p0 = kb; p0 < ke; p0 += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = p0 + u;
      uint16_t *buf = rows[u & 1];  // one wave: the step before last has read it
      if (lane < SR * OCT) *reinterpret_cast<u32x4 *>(buf + 8 * lane) = st[u].x & st[u].in;
      u32x4 a[2][MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const float dv[4] = {st[u].d[m].x, st[u].d[m].y, st[u].d[m].z, st[u].d[m].w};
        const uint32_t c = st[u].c[m];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float v = p < ke ? (c & (4u << (8 * j)) ? dv[j] : kLeak * dv[j]) : 0.0f;
          bias[m] += v;
          // at its column, in the row of the window that held the maximum
          const uint32_t w = static_cast<uint32_t>(bf16_rne(v)) << (c >> (8 * j) & 1u) * 16;
          const bool low = c & (2u << (8 * j));
          a[0][m][j] = low ? 0u : w;
          a[1][m][j] = low ? w : 0u;
        }
      }
      __syncthreads();
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const u32x4 o = *reinterpret_cast<const u32x4 *>(buf + at0[t] + h * SW);
          const uint32_t e = *reinterpret_cast<const uint32_t *>(buf + edge[t] + h * SW);
          const u32x4 right = octet_right(o, e), left = octet_left(o, e);
          const bf16x8 bb = __builtin_bit_cast(bf16x8, dxc[t] < 0 ? right : dxc[t] > 0 ? left : o);
#pragma unroll
          for (int m = 0; m < MT; ++m)
            acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[h][m]), bb, acc[m][t], 0, 0, 0);
        }
      __builtin_amdgcn_sched_barrier(0);
      if (u & 1) {  // a line of each row of dy
        load(p + U - 1, st[u - 1]);
        load(p + U, st[u]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  float *out = ws + static_cast<size_t>(z) * COUT * (N + 1);
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    bias[m] += __shfl_xor(bias[m], 16);
    bias[m] += __shfl_xor(bias[m], 32);
    if (lane < 16) out[COUT * N + 16 * m + r16] = bias[m];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int c = t * 16 + r16;
      if (c >= N) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) out[(16 * m + (lane >> 4) * 4 + r) * N + c] = acc[m][t][r];
    }
  }
}

// 3x3 convolution of a layer as a product over k = channel*9 + tap (padding
// 1): forward (BWD false; bias, leaky ReLU, of the bf16 output its 2x2 maximum
// `pool` and, where a backward pass follows, the windows' codes) or the
// gradient of the layer's input (BWD true: CI the layer's output channels, x
// their bf16 gradients, the stencil mirrored, float32 output dx). Four waves share a patch of the input in LDS, with its border
// (zeros outside the image); each takes all output channels of 2 rows x 32
// columns. A lane gathers its pixel's eight operands of a matrix instruction
// from the patch, at offsets (in elements) that a table in LDS holds for
// every k, and reads the weights [CO][K] as the instruction takes them. The
// gathers bind it: eight 2-byte LDS reads per 16 pixels and 32 k serve CO/16
// instructions. Accumulators stay in vector registers (two waves per SIMD
// asked for: with one, the compiler keeps them in the other half of the file
// and moves them for every addition). 64 samples, layers one to four forward
// with the pooling: 48, 41, 19 and 19 us; backward, layers two to four: 40, 27
// and 14 (181 and 147 us a layer through the general product, which forms every
// element's index anew, and a pooling of its own).
// SPLIT, for a batch whose pixels and channels are fewer than 256 tiles of 64 x
// 64: `per` matrix instructions in a row make a partial sum, and the partial
// sums are added in order (the sums of a product split over k). As most CUs
// would have no block, a block takes 2 rows x 16 columns, and its four waves
// every fourth partial sum. One sample, layers two to four: 5.1, 4.8 and
// 7.4 us (5.4, 6.1 and 10.4 with one wave for all of them; 7.4, 10.4 and 14.3 as
// blocks of four waves' 2 x 32 pixels).
template <int CI, int CO, int H, int W, bool SPLIT>
struct ConvGeo {
  static constexpr int K = CI * 9, STEPS = (K + 31) / 32, MT = CO / 16;
  static constexpr int WAVES = SPLIT ? 1 : 4, TC = SPLIT ? 1 : 2, WC = 16 * TC;  // waves side by side; a wave's columns
  static constexpr int COLS = SPLIT ? WC : W < 128 ? W : 128, WX = COLS / WC, RB = 2 * (WAVES / WX);
  static constexpr int XB = W / COLS, YB = (H + RB - 1) / RB;
  static constexpr int PR = RB + 2, STRIDE = COLS + 16;  // patch rows; columns with eight on either side
  static constexpr int OUT = WAVES * CO * 2 * WC;        // elements of the block's output tile
  static constexpr int ELEMS = CI * PR * STRIDE > OUT ? CI * PR * STRIDE : OUT;
  static constexpr int PS = 2 * WC + 4;                  // floats of a channel in a partial sum's tile
};

template <int CI, int CO, int H, int W, bool BWD, bool SPLIT>
__global__ __launch_bounds__(256, 2) void conv_kernel(const uint16_t *__restrict__ x, const uint16_t *__restrict__ w,
                                                   const float *__restrict__ bias, uint16_t *__restrict__ pool,
                                                   uint8_t *__restrict__ code, float *__restrict__ dx, int per) {
  using G = ConvGeo<CI, CO, H, W, SPLIT>;
  constexpr int K = G::K, MT = G::MT, HW = H * W, NT = 256, T = 2 * G::TC, WC = G::WC;
  __shared__ __align__(16) uint16_t patch[G::ELEMS];
  __shared__ __align__(16) uint16_t offs[G::STEPS * 32];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r16 = lane & 15, g8 = (lane >> 4) * 8;
  const int x0 = (blockIdx.x % G::XB) * G::COLS, y0 = (blockIdx.x / G::XB) * G::RB;
  const size_t b = blockIdx.y;
  for (int k = tid; k < G::STEPS * 32; k += NT) {
    const int kk = k < K ? k : 0, ci = kk / 9, r = kk - 9 * ci;
    const int row = BWD ? 2 - r / 3 : r / 3, col = BWD ? 1 - r % 3 : r % 3 - 1;
    offs[k] = static_cast<uint16_t>((ci * G::PR + row) * G::STRIDE + col + 8);
  }
  {
    constexpr int OCT = G::STRIDE / 8, ITEMS = CI * G::PR * OCT, PT = (ITEMS + NT - 1) / NT;
    const uint16_t *xb = x + b * CI * HW;
    u32x4 v[PT];
    bool in[PT];
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      const int i = min(tid + NT * j, ITEMS - 1), o = i % OCT, t = i / OCT, pr = t % G::PR, ci = t / G::PR;
      const int xx = x0 + 8 * (o - 1), yy = y0 - 1 + pr;
      in[j] = xx >= 0 && xx < W && yy >= 0 && yy < H;
      // the network's input is the caller's, aligned to its elements only
      v[j] = __builtin_bit_cast(u32x4, *reinterpret_cast<const u16x8u *>(xb + (in[j] ? ci * HW + yy * W + xx : 0)));
    }
#pragma unroll
    for (int j = 0; j < PT; ++j)
      if (tid + NT * j < ITEMS) *reinterpret_cast<u32x4 *>(patch + 8 * (tid + NT * j)) = in[j] ? v[j] : u32x4{};
  }
  __syncthreads();
  const int sw = SPLIT ? 0 : wave, wx = (sw % G::WX) * WC, wy = (sw / G::WX) * 2;  // the wave's pixels in the block
  f4 acc[T][MT];
  auto clear = [&] {
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[t][m] = f4{0.f, 0.f, 0.f, 0.f};
  };
  clear();
  const uint16_t *base[T];  // tile t: row t / TC, columns 16 (t % TC) ...
#pragma unroll
  for (int t = 0; t < T; ++t) base[t] = patch + (wy + t / G::TC) * G::STRIDE + wx + 16 * (t % G::TC) + r16;
  u16x8 next[MT];  // the weights of the next 32 k, in flight during a step
  auto weights = [&](int c) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const uint16_t *row = w + (16 * m + r16) * K + 32 * c + g8;
      if constexpr (K % 32 == 0) {
        next[m] = *reinterpret_cast<const u16x8 *>(row);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) next[m][j] = 32 * c + g8 + j < K ? row[j] : static_cast<uint16_t>(0);
      }
    }
  };
  u16x8 o_next;
  auto ahead = [&](int c) {
    weights(min(c, G::STEPS - 1));
    o_next = *reinterpret_cast<const u16x8 *>(offs + 32 * min(c, G::STEPS - 1) + g8);
  };
  auto step = [&](int c, int then) {  // step c, its operands in flight; `then` is the wave's next
    bf16x8 a[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) a[m] = __builtin_bit_cast(bf16x8, next[m]);
    const u16x8 o = o_next;
    if (G::STEPS > 1) ahead(then);
#pragma unroll
    for (int t = 0; t < T; ++t) {
      u16x8 e;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        e[j] = base[t][o[j]];
        if (K % 32 != 0 && 32 * c + g8 + j >= K) e[j] = 0;
      }
      const bf16x8 bv = __builtin_bit_cast(bf16x8, e);
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], bv, acc[t][m], 0, 0, 0);
    }
  };
  const int row4 = (lane >> 4) * 4;
  constexpr int E = SPLIT ? CO * 2 * WC / NT : 1;  // outputs that a thread adds up
  float total[E] = {};
  if constexpr (SPLIT) {
    __shared__ float part[4][CO * G::PS];  // a wave's partial sum: [channel][2][WC]
    ahead(wave * per);
    for (int c0 = 0; c0 < G::STEPS; c0 += 4 * per) {
      const int cb = c0 + wave * per, ce = min(cb + per, G::STEPS);
      clear();
      for (int c = cb; c < ce; ++c) step(c, c + 1 < ce ? c + 1 : cb + 4 * per);
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int r = 0; r < 4; ++r) part[wave][(16 * m + row4 + r) * G::PS + WC * t + r16] = acc[t][m][r];
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (c0 + k * per < G::STEPS)
#pragma unroll
          for (int i = 0; i < E; ++i) {
            const int at = tid + NT * i;
            total[i] += part[k][at / (2 * WC) * G::PS + at % (2 * WC)];
          }
      __syncthreads();
    }
  } else {
    ahead(0);
    for (int c = 0; c < G::STEPS; ++c) step(c, c + 1);
  }
  if constexpr (BWD) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int yy = y0 + wy + t / G::TC, xx = x0 + wx + 16 * (t % G::TC) + r16;
      if (yy >= H) continue;
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) dx[(b * CO + 16 * m + row4 + r) * HW + yy * W + xx] = acc[t][m][r];
    }
  } else {
    // the tile through LDS, so that the stores and the pooling take octets
    __syncthreads();
    uint16_t *out = patch + sw * (CO * 2 * WC);  // [CO][2][WC]
    if constexpr (SPLIT) {
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const int at = tid + NT * i;
        out[at] = bf16_rne(leaky(total[i] + bias[at / (2 * WC)]));
      }
    } else {
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int co = 16 * m + row4 + r;
            out[co * 2 * WC + WC * (t / G::TC) + 16 * (t % G::TC) + r16] = bf16_rne(leaky(acc[t][m][r] + bias[co]));
          }
    }
    __syncthreads();
    const int yy = y0 + wy, col = 8 * (lane % (WC / 8)), xx = x0 + wx + col;
#pragma unroll
    for (int i = 0; i < CO / (512 / WC); ++i) {
      if (SPLIT && i != wave) continue;
      const int co = 512 / WC * i + lane / (WC / 8);
      const u16x8 top = *reinterpret_cast<const u16x8 *>(out + co * 2 * WC + col);
      const u16x8 low = *reinterpret_cast<const u16x8 *>(out + co * 2 * WC + WC + col);
      if (yy + 1 >= H) continue;
      const size_t at = (b * CO + co) * (H / 2) * (W / 2) + (yy / 2) * (W / 2) + xx / 2;
      typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
      u16x4 mx;
      uint32_t codes = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float v = bf16_f(top[2 * j]);
        v = fmaxf(v, bf16_f(top[2 * j + 1]));
        v = fmaxf(v, bf16_f(low[2 * j]));
        v = fmaxf(v, bf16_f(low[2 * j + 1]));
        mx[j] = bf16_rne(v);
        codes |= pool_code(top[2 * j], top[2 * j + 1], low[2 * j], low[2 * j + 1]) << (8 * j);
      }
      *reinterpret_cast<u16x4 *>(pool + at) = mx;
      if (code) *reinterpret_cast<uint32_t *>(code + at) = codes;
    }
  }
}

// End of the network, 16 samples per workgroup: h = leaky(sum over splits of
// ws[z][unit][sample] + b1) as bf16 (the first fully connected layer's
// product, split over k), out = w2 h + b2. The sum runs over the splits in
// order, so 1024 threads stage 64 splits at a time for the 256 that add them.
// One sample 6.4 us, 64 samples 8.6 (9.1 and 9.8 with the second layer apart).
__global__ __launch_bounds__(1024) void head_kernel(const float *__restrict__ ws, int splits,
                                                    const float *__restrict__ b1, const uint16_t *__restrict__ w2,
                                                    const float *__restrict__ b2, uint16_t *__restrict__ h1,
                                                    float *__restrict__ out, int B) {
  constexpr int C = 64;  // splits at a time
  __shared__ float part[C][256];  // [unit][sample] of a split
  __shared__ __align__(16) uint16_t hs[16][16];  // [sample][unit]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r16 = lane & 15, g8 = (lane >> 4) * 8;
  const int s0 = blockIdx.x * 16;
  const int o = tid & 255, g = tid >> 8;  // output (unit o / 16, sample o % 16), quarter of the splits
  const size_t at = static_cast<size_t>(o >> 4) * B + min(s0 + (o & 15), B - 1);
  float v = 0.0f;
  for (int z0 = 0; z0 < splits; z0 += C) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < C / 4; ++j)
      part[g + 4 * j][o] = ws[static_cast<size_t>(min(z0 + g + 4 * j, splits - 1)) * kH1 * B + at];
    __syncthreads();
    if (tid < 256) {
      const int n = min(C, splits - z0);
      if (n == C) {
#pragma unroll
        for (int z = 0; z < C; ++z) v += part[z][tid];
      } else {
        for (int z = 0; z < n; ++z) v += part[z][tid];
      }
    }
  }
  if (tid < 256) {
    const int u = tid >> 4, smp = tid & 15;
    const uint16_t h = bf16_rne(leaky(v + b1[u]));
    hs[smp][u] = h;
    if (s0 + smp < B) h1[static_cast<size_t>(s0 + smp) * kH1 + u] = h;
  }
  __syncthreads();
  if (wave != 0) return;
  // out[o][sample]: 16 units of the 32 a matrix instruction multiplies
  u16x8 a = {}, b = {};
  if (g8 < 16) {
    if (r16 < kOut) a = *reinterpret_cast<const u16x8 *>(w2 + r16 * kH1 + g8);
    b = *reinterpret_cast<const u16x8 *>(&hs[r16][g8]);
  }
  f4 acc = {0.f, 0.f, 0.f, 0.f};
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
  if (lane < 16 && s0 + r16 < B) {
#pragma unroll
    for (int o = 0; o < kOut; ++o) out[static_cast<size_t>(s0 + r16) * kOut + o] = acc[o] + b2[o];
  }
}

// The weights of layers two to four as the input gradients' products take
// them, wt[ci][co*9 + tap] = w[co][ci*9 + tap], one layer after the other.
constexpr int kWtAt[5] = {0, 0, 32 * 32 * 9, 32 * 32 * 9 + 32 * 64 * 9, 32 * 32 * 9 + 32 * 64 * 9 + 64 * 64 * 9};
__global__ __launch_bounds__(256) void transpose_weights(const uint16_t *__restrict__ w2,
                                                         const uint16_t *__restrict__ w3,
                                                         const uint16_t *__restrict__ w4, uint16_t *__restrict__ wt) {
  int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= kWtAt[4]) return;
  const int l = i < kWtAt[2] ? 1 : i < kWtAt[3] ? 2 : 3;
  const int cout = kConv[l].cout, cin = kConv[l].cin;
  const uint16_t *w = l == 1 ? w2 : l == 2 ? w3 : w4;
  wt += kWtAt[l];
  i -= kWtAt[l];
  const int co = i / (cin * 9), q = i - co * cin * 9, ci = q / 9, r = q - 9 * ci;
  wt[(ci * cout + co) * 9 + r] = w[i];
}

// Sums over the splits of a product, in a fixed order, of two products in one
// launch: 16 outputs per block, each summed by G threads over interleaved
// splits (z = g, g + G, ...) and their G partials added in order. Bound by the
// latency of a thread's loads, which are independent: 64 threads per output
// from 256 splits on (2002 splits of 576 outputs 5 us, 720 of 9216 11 us; 38 and
// 16 with 16 threads), 16 below, where most of 64 would find none (180 and 44
// splits: 5.5 us, a launch).
struct Partials {
  const float *ws;  // [splits][MN], `stride` from one split to the next
  float *out;
  int splits, MN, stride;
};
template <int G>
__global__ __launch_bounds__(16 * G) void reduce_splits(Partials a, Partials b) {
  const int o = threadIdx.x & 15, g = threadIdx.x >> 4, blocks_a = (a.MN + 15) / 16;
  const Partials p = static_cast<int>(blockIdx.x) < blocks_a ? a : b;
  const int i = (blockIdx.x - (static_cast<int>(blockIdx.x) < blocks_a ? 0 : blocks_a)) * 16 + o;
  float s = 0.0f;
  if (i < p.MN) {
#pragma unroll 8
    for (int z = g; z < p.splits; z += G) s += p.ws[static_cast<size_t>(z) * p.stride + i];
  }
  __shared__ float part[G][17];
  part[g][o] = s;
  __syncthreads();
  if (g == 0 && i < p.MN) {
    float t = part[0][o];
#pragma unroll 16
    for (int k = 1; k < G; ++k) t += part[k][o];
    p.out[i] = t;
  }
}
hipError_t launch_reduce(Partials a, Partials b, hipStream_t s) {
  const dim3 grid((a.MN + 15) / 16 + (b.MN + 15) / 16);
  if (std::max(a.splits, b.splits) >= 256)
    hipLaunchKernelGGL(reduce_splits<64>, grid, dim3(1024), 0, s, a, b);
  else
    hipLaunchKernelGGL(reduce_splits<16>, grid, dim3(256), 0, s, a, b);
  return hipGetLastError();
}

// Loss over targets t[b] = {offset, tolerance} (output units):
// Huber(offset error, delta 0.25) + 0.2 * BCE(confidence logit, |error| < tolerance),
// mean over the batch, with its gradient g = dL/d(out) / B, and the backward
// pass of the second fully connected layer: the gradients of its weights w
// (dw, operands rounded to bf16 as in the other layers' products) and bias
// (db), of its input h (gh) and of the first layer's bias (db1, with the slope
// of h). One workgroup: the sums run over a batch of tens of samples, and what
// it costs is its launch: 4.7 us, 29 with a kernel for the loss, each product,
// its split sum and each bias sum.
__global__ __launch_bounds__(256) void loss_kernel(const float *__restrict__ out, const float *__restrict__ tgt,
                                                   const uint16_t *__restrict__ h, const uint16_t *__restrict__ w,
                                                   float *g, float *__restrict__ loss, float *__restrict__ dw,
                                                   float *__restrict__ db, float *__restrict__ gh,
                                                   float *__restrict__ db1, int B) {
  static_assert(kH1 == 16 && kOut == 2, "a thread per unit and sixteenth of the batch");
  __shared__ float red[256];
  float l = 0.0f;
  for (int b = threadIdx.x; b < B; b += blockDim.x) {
    const float e = out[2 * b] - tgt[2 * b];
    const float delta = 0.25f;
    const float ae = fabsf(e);
    const float hub = ae < delta ? 0.5f * e * e / delta : ae - 0.5f * delta;
    const float dh = ae < delta ? e / delta : (e > 0 ? 1.0f : -1.0f);
    const float y = ae < tgt[2 * b + 1] ? 1.0f : 0.0f;
    const float z = out[2 * b + 1];
    const float p = 1.0f / (1.0f + expf(-z));
    const float bce = fmaxf(z, 0.0f) - z * y + log1pf(expf(-fabsf(z)));
    l += hub + 0.2f * bce;
    g[2 * b] = dh / B;
    g[2 * b + 1] = 0.2f * (p - y) / B;
  }
  red[threadIdx.x] = l;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) *loss = red[0] / B;
  const int k = threadIdx.x & 15, q = threadIdx.x >> 4;
  const float w0 = bf16_f(w[k]), w1 = bf16_f(w[kH1 + k]);
  float s[5] = {};  // dw of the two outputs, db1; db of the two outputs
  for (int b = q; b < B; b += 16) {
    const float d0 = g[2 * b], d1 = g[2 * b + 1];
    const float q0 = bf16_f(bf16_rne(d0)), q1 = bf16_f(bf16_rne(d1)), hv = bf16_f(h[b * kH1 + k]);
    const float v = w0 * q0 + w1 * q1;
    gh[b * kH1 + k] = v;
    s[0] += q0 * hv;
    s[1] += q1 * hv;
    s[2] += hv > 0.0f ? v : kLeak * v;
    s[3] += d0;
    s[4] += d1;
  }
  __shared__ float part[5][16][17];
#pragma unroll
  for (int j = 0; j < 5; ++j) part[j][q][k] = s[j];
  __syncthreads();
  if (q >= 5 || (q >= 3 && k > 0)) return;
  float t = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; ++i) t += part[q][i][k];
  if (q < 2) dw[q * kH1 + k] = t;
  else if (q == 2) db1[k] = t;
  else db[q - 3] = t;
}

// Global gradient norm: per-block sums of squares, then one block sums them
// in a fixed order and writes the clipping factor min(1, clip / norm) (1
// when clip <= 0) and the norm.
constexpr int kNormBlocks = 256;

__global__ __launch_bounds__(256) void sumsq_kernel(const float *__restrict__ g, int n, float *__restrict__ part) {
  __shared__ float red[256];
  float s = 0.0f;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += kNormBlocks * 256) s += g[i] * g[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void clip_factor_kernel(const float *__restrict__ part, float clip,
                                                          float *__restrict__ out) {
  __shared__ float red[256];
  red[threadIdx.x] = threadIdx.x < kNormBlocks ? part[threadIdx.x] : 0.0f;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const float norm = sqrtf(red[0]);
    out[0] = (clip > 0.0f && norm > clip) ? clip / norm : 1.0f;
    out[1] = norm;
  }
}

__global__ void adam_kernel(float *__restrict__ p, uint16_t *__restrict__ p16, const float *__restrict__ g,
                            float *__restrict__ m, float *__restrict__ v, int n, float lr, float b1, float b2,
                            float c1, float c2, float eps, const float *__restrict__ scale) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i] * scale[0];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  p[i] = pi;
  p16[i] = bf16_rne(pi);
}

// The parameters, each at its aligned offset, one after the other.
constexpr int kParams = 12;
struct Packing {
  int off[kParams], at[kParams];  // of parameter i in p and in out
};
__global__ __launch_bounds__(256) void pack_params(const float *__restrict__ p, float *__restrict__ out, Packing pk,
                                                   int count) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  int from = i;
#pragma unroll
  for (int k = 0; k < kParams; ++k)
    if (i >= pk.at[k]) from = pk.off[k] + i - pk.at[k];
  out[i] = p[from];
}

__global__ void to_bf16(const float *__restrict__ p, uint16_t *__restrict__ q, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) q[i] = bf16_rne(p[i]);
}

// Sinogram [N][w] (transmission) -> features [2][180][256] bf16: the mean
// of -log(max(v, 1e-6)) over each cell of angle rows x detector columns,
// standardised per sample; channel 1 is the map turned by 180 degrees
// (detector and angle order reversed), which puts the projections that
// mirror each other across the 0/180 degree seam (P(theta + pi, s) =
// P(theta, -s)) in the same rows of the two channels, shifted by twice
// the axis offset. Grid (1, 180): one block per angle cell.
// The cells' sums run row by row and column by column, a cell per thread, so
// a block of 1024 takes the logarithms of a row coalesced into LDS, 4096
// columns at a time, and the 256 owners add their columns from there. One
// thread per cell, reading its columns from memory, took 13.5 us for 1800 x
// 2048, bound by the logarithms of three waves per CU; this takes 9 to 10.
constexpr int kFeatCols = 4096, kFeatT = 1024;
__global__ __launch_bounds__(kFeatT) void features_kernel(const float *__restrict__ sino, int N, int w,
                                                          float *__restrict__ tmp) {
  __shared__ float line[2][kFeatCols];
  const int a = blockIdx.y;
  const int x = threadIdx.x;
  const int r0 = static_cast<int>(static_cast<long long>(a) * N / kFeatA);
  const int r1 = max(r0 + 1, static_cast<int>(static_cast<long long>(a + 1) * N / kFeatA));
  const int c0 = static_cast<int>(static_cast<long long>(x) * w / kFeatW);
  const int c1 = max(c0 + 1, static_cast<int>(static_cast<long long>(x + 1) * w / kFeatW));
  constexpr int PT = kFeatCols / kFeatT;
  // a step takes as many whole rows as fit, or a part of one row
  const int rps = max(1, kFeatCols / w), nseg = (w + kFeatCols - 1) / kFeatCols;
  const int steps = nseg > 1 ? (r1 - r0) * nseg : (r1 - r0 + rps - 1) / rps;
  const size_t last = static_cast<size_t>(r1) * w - 1;  // of the cell's samples
  float v[PT];
  auto fetch = [&](int k) {
    const size_t at = static_cast<size_t>(r0 + (nseg > 1 ? k / nseg : k * rps)) * w + (nseg > 1 ? (k % nseg) * kFeatCols : 0);
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      const size_t i = at + x + kFeatT * j;
      v[j] = sino[i < last ? i : last];
    }
  };
  fetch(0);
  float s = 0.0f;
  for (int k = 0; k < steps; ++k) {
    float *buf = line[k & 1];
#pragma unroll
    for (int j = 0; j < PT; ++j) buf[x + kFeatT * j] = -logf(fmaxf(v[j], 1e-6f));
    if (k + 1 < steps) fetch(k + 1);
    __syncthreads();
    if (x >= kFeatW) continue;
    if (nseg > 1) {
      const int b = (k % nseg) * kFeatCols;
      for (int c = max(c0, b); c < min(c1, b + kFeatCols); ++c) s += buf[c - b];
    } else {
      const int rows = min(rps, r1 - r0 - k * rps);
      for (int r = 0; r < rows; ++r)
        for (int c = c0; c < c1; ++c) s += buf[r * w + c];
    }
  }
  if (x < kFeatW) tmp[a * kFeatW + x] = s / static_cast<float>((r1 - r0) * (c1 - c0));
}

// Mean and standard deviation of the 180 x 256 features, then the two
// standardised bf16 channels. Every block of 1024 threads forms the sums for
// itself (a thread's 12 float4 loads in flight together, partial sums reduced
// in a fixed order) and writes 1024 features: one block doing all of it, a
// load at a time, took 16 us; this takes 4.6.
__global__ __launch_bounds__(1024) void standardise_kernel(const float *__restrict__ tmp, uint16_t *__restrict__ feat) {
  __shared__ float red[1024], red2[1024];
  constexpr int n = kFeatA * kFeatW, Q = n / 4, PT = (Q + 1023) / 1024;
  static_assert(n % 1024 == 0, "whole blocks of features");
  const float4 *t4 = reinterpret_cast<const float4 *>(tmp);
  float4 q[PT];
#pragma unroll
  for (int j = 0; j < PT; ++j) q[j] = t4[min(static_cast<int>(threadIdx.x) + 1024 * j, Q - 1)];
  const int i = blockIdx.x * 1024 + threadIdx.x;
  const float mine = tmp[i];
  float s = 0.0f, s2 = 0.0f;
#pragma unroll
  for (int j = 0; j < PT; ++j)
    if (static_cast<int>(threadIdx.x) + 1024 * j < Q) {
      const float4 v = q[j];
      s += (v.x + v.y) + (v.z + v.w);
      s2 += (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w);
    }
  red[threadIdx.x] = s;
  red2[threadIdx.x] = s2;
  __syncthreads();
  for (int o = 512; o > 0; o >>= 1) {
    if (static_cast<int>(threadIdx.x) < o) {
      red[threadIdx.x] += red[threadIdx.x + o];
      red2[threadIdx.x] += red2[threadIdx.x + o];
    }
    __syncthreads();
  }
  const float mean = red[0] / n;
  const float var = fmaxf(red2[0] / n - mean * mean, 1e-12f);
  const float inv = 1.0f / sqrtf(var);
  const int a = i / kFeatW, x = i - a * kFeatW;
  const float v = (mine - mean) * inv;
  feat[i] = bf16_rne(v);
  feat[n + (kFeatA - 1 - a) * kFeatW + (kFeatW - 1 - x)] = bf16_rne(v);
}

hipError_t launch_features(const float *d_sino, int N, int w, float *d_tmp, uint16_t *d_x, hipStream_t s) {
  hipLaunchKernelGGL(features_kernel, dim3(1, kFeatA), dim3(kFeatT), 0, s, d_sino, N, w, d_tmp);
  hipLaunchKernelGGL(standardise_kernel, dim3(kFeatA * kFeatW / 1024), dim3(1024), 0, s, d_tmp, d_x);
  return hipGetLastError();
}

struct Param {
  size_t off, n;
};

}  // namespace cnn
}  // namespace ctas

struct ctas_cnn {
  int device = 0;
  hipStream_t stream = nullptr;
  std::vector<ctas::cnn::Param> prm;  // w1 b1 w2 b2 w3 b3 w4 b4 wf1 bf1 wf2 bf2
  size_t nparam = 0;
  float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
  uint16_t *p16 = nullptr, *wt = nullptr;  // bf16 weights; those of layers two to four, transposed
  int step = 0;
  int cap = 0;  // batch capacity of the activation buffers
  uint16_t *pool[4] = {}, *h1 = nullptr;
  uint8_t *code[4] = {};  // of the pooling's windows, for the backward pass
  uint16_t *gact = nullptr;  // bf16 gradient of a layer's pre-activation (layers two to four)
  float *out = nullptr, *gout = nullptr, *gh1 = nullptr, *gf = nullptr, *gbig2 = nullptr;
  float *ws = nullptr;
  size_t ws_cap = 0;
  float *loss = nullptr;
  // pinned: a prediction's two outputs and a batch's loss, written by their
  // kernels; null where none was to be had (they are copied then)
  float *host = nullptr;
  float *ftmp = nullptr;
  uint16_t *xin = nullptr;  // features of one sinogram (prediction)
  float *norm = nullptr;    // gradient-norm partials, clip factor, norm
};

namespace ctas {
namespace cnn {
namespace {

int alloc(void **p, size_t bytes) {
  if (hipMalloc(p, std::max<size_t>(bytes, 256)) != hipSuccess) {
    *p = nullptr;
    return fail(CTAS_E_NOMEM, "CNN allocation of " + std::to_string(bytes) + " bytes failed");
  }
  return CTAS_OK;
}

void release_batch(ctas_cnn *n) {
  for (int l = 0; l < 4; ++l) {
    if (n->pool[l]) (void)hipFree(n->pool[l]);
    if (n->code[l]) (void)hipFree(n->code[l]);
    n->pool[l] = nullptr;
    n->code[l] = nullptr;
  }
  void *ptrs[] = {n->h1, n->out, n->gout, n->gh1, n->gf, n->gact, n->gbig2};
  for (void *q : ptrs)
    if (q) (void)hipFree(q);
  n->h1 = nullptr;
  n->gact = nullptr;
  n->out = n->gout = n->gh1 = n->gf = n->gbig2 = nullptr;
  n->cap = 0;
}

int ensure_batch(ctas_cnn *n, int B) {
  if (B <= n->cap) return CTAS_OK;
  CTAS_HIP_TRY(hipStreamSynchronize(n->stream));
  release_batch(n);
  size_t big = 0;
  for (int l = 0; l < 4; ++l) {
    const Layer &L = kConv[l];
    const size_t q = static_cast<size_t>(B) * L.cout * (L.H / 2) * (L.W / 2);
    if (int rc = alloc(reinterpret_cast<void **>(&n->pool[l]), q * 2)) return rc;
    if (int rc = alloc(reinterpret_cast<void **>(&n->code[l]), q)) return rc;
    if (l > 0) big = std::max(big, static_cast<size_t>(B) * std::max(L.cin, L.cout) * L.H * L.W);
  }
  if (int rc = alloc(reinterpret_cast<void **>(&n->h1), static_cast<size_t>(B) * kH1 * 2)) return rc;
  if (int rc = alloc(reinterpret_cast<void **>(&n->out), static_cast<size_t>(B) * kOut * 4)) return rc;
  if (int rc = alloc(reinterpret_cast<void **>(&n->gout), static_cast<size_t>(B) * kOut * 4)) return rc;
  if (int rc = alloc(reinterpret_cast<void **>(&n->gh1), static_cast<size_t>(B) * kH1 * 4)) return rc;
  if (int rc = alloc(reinterpret_cast<void **>(&n->gf), static_cast<size_t>(B) * kF * 4)) return rc;
  if (int rc = alloc(reinterpret_cast<void **>(&n->gact), big * 2)) return rc;
  if (int rc = alloc(reinterpret_cast<void **>(&n->gbig2), big * 4)) return rc;
  n->cap = B;
  return CTAS_OK;
}

int ensure_ws(ctas_cnn *n, size_t floats) {
  if (floats <= n->ws_cap) return CTAS_OK;
  CTAS_HIP_TRY(hipStreamSynchronize(n->stream));
  if (n->ws) (void)hipFree(n->ws);
  n->ws = nullptr;
  n->ws_cap = 0;
  if (int rc = alloc(reinterpret_cast<void **>(&n->ws), floats * 4)) return rc;
  n->ws_cap = floats;
  return CTAS_OK;
}

const uint16_t *W16(const ctas_cnn *n, int i) { return n->p16 + n->prm[i].off; }
const float *P32(const ctas_cnn *n, int i) { return n->p + n->prm[i].off; }
float *G32(const ctas_cnn *n, int i) { return n->g + n->prm[i].off; }

// Splits of the reduction for a product whose C tiles alone would not fill
// the chip (inference on a single sinogram); 1 when they do.
int forward_splits(int M, int N, int K) {
  const int tiles = ((M + kBT - 1) / kBT) * ((N + kBT - 1) / kBT);
  if (tiles >= 256) return 1;
  return std::max(1, std::min((256 + tiles - 1) / tiles, K / 64));
}

// Convolution layer l with its pooling. The sums are those of a product
// split over k where one of 64x64 tiles would not fill the chip. `codes`: a
// backward pass follows.
template <int L, int CI, int CO, int H, int W>
hipError_t conv_forward(ctas_cnn *n, const uint16_t *x, int B, bool codes) {
  using G = ConvGeo<CI, CO, H, W, false>;
  using S = ConvGeo<CI, CO, H, W, true>;
  const int splits = forward_splits(CO, B * H * W, G::K), per = (G::STEPS + splits - 1) / splits;
  uint8_t *code = codes ? n->code[L] : nullptr;
  if constexpr (G::STEPS > 1) {
    if (per < G::STEPS) {
      hipLaunchKernelGGL((conv_kernel<CI, CO, H, W, false, true>), dim3(S::XB * S::YB, B), dim3(256), 0, n->stream, x,
                         W16(n, 2 * L), P32(n, 2 * L + 1), n->pool[L], code, nullptr, per);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((conv_kernel<CI, CO, H, W, false, false>), dim3(G::XB * G::YB, B), dim3(256), 0, n->stream, x, W16(n, 2 * L),
                     P32(n, 2 * L + 1), n->pool[L], code, nullptr, per);
  return hipGetLastError();
}

// Gradient of the input of layer l into gbig2.
template <int L, int CIN, int COUT, int H, int W>
hipError_t conv_input_grad(ctas_cnn *n, const uint16_t *g, int B) {
  using G = ConvGeo<COUT, CIN, H, W, false>;
  hipLaunchKernelGGL((conv_kernel<COUT, CIN, H, W, true, false>), dim3(G::XB * G::YB, B), dim3(256), 0, n->stream, g,
                     n->wt + kWtAt[L], nullptr, nullptr, nullptr, n->gbig2, G::STEPS);
  return hipGetLastError();
}

// `out` [B][2]: device or pinned memory.
int forward(ctas_cnn *n, const uint16_t *x, int B, bool codes, float *out) {
  hipStream_t s = n->stream;
  CTAS_HIP_TRY((conv_forward<0, 2, 32, 180, 256>(n, x, B, codes)));
  CTAS_HIP_TRY((conv_forward<1, 32, 32, 90, 128>(n, n->pool[0], B, codes)));
  CTAS_HIP_TRY((conv_forward<2, 32, 64, 45, 64>(n, n->pool[1], B, codes)));
  CTAS_HIP_TRY((conv_forward<3, 64, 64, 22, 32>(n, n->pool[2], B, codes)));
  int splits = forward_splits(kH1, B, kF);
  const int chunk = ((kF + splits - 1) / splits + kKS - 1) & ~(kKS - 1);
  if (int rc = ensure_ws(n, static_cast<size_t>(splits) * kH1 * B)) return rc;
  CTAS_HIP_TRY(gemm(DenseA{W16(n, 8), kF}, ActB{n->pool[3], kF}, StorePartial{n->ws, kH1, B}, kH1, B, kF, s, splits));
  splits = (kF + chunk - 1) / chunk;  // those that hold any k
  hipLaunchKernelGGL(head_kernel, dim3((B + 15) / 16), dim3(1024), 0, s, n->ws, splits, P32(n, 9), W16(n, 10),
                     P32(n, 11), n->h1, out, B);
  CTAS_HIP_TRY(hipGetLastError());
  return CTAS_OK;
}

// Weight gradient of the first fully connected layer on B samples: K is split
// (and the splits summed in a fixed order) only where the batch is large.
int dense_weight_grad(ctas_cnn *n, int B, float *dst) {
  const GradFlatA fa{n->gh1, n->h1, kH1};
  const ActBT fb{n->pool[3], kF};
  int splits = std::max(1, std::min(2048, B / 1024));
  if (splits == 1) {
    CTAS_HIP_TRY(gemm(fa, fb, StorePartial{dst, kH1, kF}, kH1, kF, B, n->stream));
    return CTAS_OK;
  }
  if (int rc = ensure_ws(n, static_cast<size_t>(splits) * kH1 * kF)) return rc;
  const int chunk = ((B + splits - 1) / splits + kKS - 1) & ~(kKS - 1);
  CTAS_HIP_TRY(gemm(fa, fb, StorePartial{n->ws, kH1, kF}, kH1, kF, B, n->stream, splits));
  splits = (B + chunk - 1) / chunk;
  CTAS_HIP_TRY(launch_reduce({n->ws, dst, splits, kH1 * kF, kH1 * kF}, {}, n->stream));
  return CTAS_OK;
}

// Gradients of a convolution layer's weights and bias on B samples, and of its
// pre-activation (gact), from that of its pooled output.
template <int L, int CIN, int COUT, int H, int W>
int conv_weight_grad(ctas_cnn *n, const float *gpool, const uint16_t *in, int B) {
  constexpr int N = CIN * 9;
  // a workgroup per CU, with four steps or more for each wave (second layer 43
  // us; 49 with two workgroups per CU)
  const int K = B * H * W;
  int splits = std::max(1, std::min(256 / (CIN / 16), K / 512));
  const int chunk = ((K + splits - 1) / splits + 127) & ~127;
  splits = (K + chunk - 1) / chunk;
  const size_t bias_at = static_cast<size_t>(splits) * COUT * N;
  if (int rc = ensure_ws(n, bias_at + static_cast<size_t>(B) * COUT)) return rc;
  hipLaunchKernelGGL(pool_bwd, dim3(COUT, B), dim3(256), 0, n->stream, n->code[L], gpool, n->gact, n->ws + bias_at,
                     COUT, H, W);
  hipLaunchKernelGGL((wgrad_kernel<CIN, COUT, H, W>), dim3(splits, CIN / 16), dim3(256), 0, n->stream, n->gact, in,
                     n->ws, K, chunk);
  CTAS_HIP_TRY(hipGetLastError());
  CTAS_HIP_TRY(launch_reduce({n->ws, G32(n, 2 * L), splits, COUT * N, COUT * N},
                             {n->ws + bias_at, G32(n, 2 * L + 1), B, COUT, COUT}, n->stream));
  return CTAS_OK;
}

// The same of the first layer, without the gradient of its pre-activation.
template <int L, int CIN, int COUT, int H, int W>
int conv_taps_grad(ctas_cnn *n, const float *gpool, const uint16_t *in, int B) {
  constexpr int MN = COUT * CIN * 9, S = MN + COUT;
  const int K = B * (H * W / 64);  // a wave takes some 1500 pixels, as in the other layers
  int splits = std::max(1, std::min(2048, K / 16));
  const int chunk = (K + splits - 1) / splits;
  splits = (K + chunk - 1) / chunk;
  if (int rc = ensure_ws(n, static_cast<size_t>(splits) * S)) return rc;
  hipLaunchKernelGGL((wgrad_taps_kernel<CIN, COUT, H, W>), dim3(splits), dim3(64), 0, n->stream, n->code[L], gpool, in,
                     n->ws, K, chunk);
  CTAS_HIP_TRY(hipGetLastError());
  CTAS_HIP_TRY(launch_reduce({n->ws, G32(n, 2 * L), splits, MN, S},
                             {n->ws + MN, G32(n, 2 * L + 1), splits, COUT, S}, n->stream));
  return CTAS_OK;
}

// From the loss's backward pass of the second fully connected layer on.
int backward(ctas_cnn *n, const uint16_t *x, int B) {
  hipStream_t s = n->stream;
  hipLaunchKernelGGL(transpose_weights, dim3((kWtAt[4] + 255) / 256), dim3(256), 0, s, W16(n, 2), W16(n, 4), W16(n, 6),
                     n->wt);
  // fc1 (ReLU on h1)
  if (int rc = dense_weight_grad(n, B, G32(n, 8))) return rc;
  CTAS_HIP_TRY(gemm(DenseAT{W16(n, 8), kF}, GradFlatB{GradFlatA{n->gh1, n->h1, kH1}}, StoreFlatDX{n->gf, kF}, kF, B,
                    kH1, s));
  // conv layers, last to first. gf = gradient of the last layer's pooled
  // output; gact = bf16 gradient of a layer's pre-activation; the gradient of
  // its input (= the previous pooled output) goes to gbig2.
  if (int rc = conv_weight_grad<3, 64, 64, 22, 32>(n, n->gf, n->pool[2], B)) return rc;
  CTAS_HIP_TRY((conv_input_grad<3, 64, 64, 22, 32>(n, n->gact, B)));
  if (int rc = conv_weight_grad<2, 32, 64, 45, 64>(n, n->gbig2, n->pool[1], B)) return rc;
  CTAS_HIP_TRY((conv_input_grad<2, 32, 64, 45, 64>(n, n->gact, B)));
  if (int rc = conv_weight_grad<1, 32, 32, 90, 128>(n, n->gbig2, n->pool[0], B)) return rc;
  CTAS_HIP_TRY((conv_input_grad<1, 32, 32, 90, 128>(n, n->gact, B)));
  return conv_taps_grad<0, 2, 32, 180, 256>(n, n->gbig2, x, B);
}

}  // namespace
}  // namespace cnn
}  // namespace ctas

using namespace ctas;
using namespace ctas::cnn;

extern "C" int ctas_cnn_create(ctas_cnn **pn, uint64_t seed) {
  if (!pn) return fail(CTAS_E_ARG, "null argument");
  *pn = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(CTAS_E_DEVICE, "no HIP device is available");
  std::unique_ptr<ctas_cnn> n(new ctas_cnn);
  CTAS_HIP_TRY(hipGetDevice(&n->device));
  CTAS_HIP_TRY(hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking));
  std::vector<std::pair<size_t, float>> shapes;  // (count, init scale)
  for (int l = 0; l < 4; ++l) {
    const size_t fan_in = static_cast<size_t>(kConv[l].cin) * 9;
    shapes.push_back({kConv[l].cout * fan_in, std::sqrt(2.0f / fan_in)});
    shapes.push_back({static_cast<size_t>(kConv[l].cout), 0.0f});
  }
  shapes.push_back({static_cast<size_t>(kH1) * kF, std::sqrt(2.0f / kF)});
  shapes.push_back({static_cast<size_t>(kH1), 0.0f});
  shapes.push_back({static_cast<size_t>(kOut) * kH1, std::sqrt(1.0f / kH1)});
  shapes.push_back({static_cast<size_t>(kOut), 0.0f});
  size_t off = 0;
  for (auto &sh : shapes) {
    n->prm.push_back({off, sh.first});
    off += (sh.first + 63) & ~static_cast<size_t>(63);
  }
  n->nparam = off;
  std::vector<float> h(off, 0.0f);
  std::mt19937_64 rng(seed);
  std::normal_distribution<float> nd(0.0f, 1.0f);
  for (size_t i = 0; i < shapes.size(); ++i)
    for (size_t k = 0; k < shapes[i].first; ++k) h[n->prm[i].off + k] = shapes[i].second * nd(rng);
  if (int rc = alloc(reinterpret_cast<void **>(&n->p), off * 4)) return rc;
  if (int rc = alloc(reinterpret_cast<void **>(&n->g), off * 4)) return rc;
  if (int rc = alloc(reinterpret_cast<void **>(&n->m), off * 4)) return rc;
  if (int rc = alloc(reinterpret_cast<void **>(&n->v), off * 4)) return rc;
  if (int rc = alloc(reinterpret_cast<void **>(&n->p16), off * 2)) return rc;
  if (int rc = alloc(reinterpret_cast<void **>(&n->wt), kWtAt[4] * 2)) return rc;
  if (int rc = alloc(reinterpret_cast<void **>(&n->loss), 256)) return rc;
  if (int rc = alloc(reinterpret_cast<void **>(&n->norm), sizeof(float) * (kNormBlocks + 2))) return rc;
  if (int rc = alloc(reinterpret_cast<void **>(&n->ftmp), sizeof(float) * kFeatA * kFeatW)) return rc;
  if (hipHostMalloc(reinterpret_cast<void **>(&n->host), 3 * sizeof(float), hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    n->host = nullptr;
  }
  CTAS_HIP_TRY(hipMemcpy(n->p, h.data(), off * 4, hipMemcpyHostToDevice));
  std::vector<float> z(off, 0.0f);
  CTAS_HIP_TRY(hipMemcpy(n->m, z.data(), off * 4, hipMemcpyHostToDevice));
  CTAS_HIP_TRY(hipMemcpy(n->v, z.data(), off * 4, hipMemcpyHostToDevice));
  CTAS_HIP_TRY(hipMemcpy(n->g, z.data(), off * 4, hipMemcpyHostToDevice));
  hipLaunchKernelGGL(to_bf16, dim3((off + 255) / 256), dim3(256), 0, n->stream, n->p, n->p16, static_cast<int>(off));
  CTAS_HIP_TRY(hipStreamSynchronize(n->stream));
  *pn = n.release();
  return CTAS_OK;
}

extern "C" int ctas_cnn_destroy(ctas_cnn *n) {
  if (!n) return CTAS_OK;
  (void)hipStreamSynchronize(n->stream);
  release_batch(n);
  void *ptrs[] = {n->p, n->g, n->m, n->v, n->p16, n->wt, n->ws, n->loss, n->ftmp, n->xin, n->norm};
  for (void *q : ptrs)
    if (q) (void)hipFree(q);
  if (n->host) (void)hipHostFree(n->host);
  (void)hipStreamDestroy(n->stream);
  delete n;
  return CTAS_OK;
}

// Parameter layout: the 12 tensors w1 b1 w2 b2 w3 b3 w4 b4 wf1 bf1 wf2 bf2
// (conv weights [cout][cin][3][3], fc weights [out][in]) packed back to back.
extern "C" int ctas_cnn_num_params(const ctas_cnn *n, int *count) {
  if (!n || !count) return fail(CTAS_E_ARG, "null argument");
  size_t c = 0;
  for (const auto &p : n->prm) c += p.n;
  *count = static_cast<int>(c);
  return CTAS_OK;
}

static int copy_params(ctas_cnn *n, float *host, const float *dev, bool to_host) {
  size_t count = 0;
  for (const auto &p : n->prm) count += p.n;
  // one after the other on the device first: most of the twelve are small, and
  // each copy has its own latency (gradients of 64 samples and their values on
  // the host: 842 us with twelve copies, 702 with one). On the network's own
  // device (copies take any) and into scratch of this call: the network's
  // workspace may be in use by another thread's prediction, and reading the
  // parameters does not change the network.
  int dev_now = -1;
  std::optional<Scratch> packed;
  if (to_host && hipGetDevice(&dev_now) == hipSuccess && dev_now == n->device) packed.emplace(count * 4);
  if (packed && packed->get()) {
    ctas::cnn::Packing pk;
    for (size_t i = 0, at = 0; i < n->prm.size(); at += n->prm[i++].n) {
      pk.off[i] = static_cast<int>(n->prm[i].off);
      pk.at[i] = static_cast<int>(at);
    }
    hipLaunchKernelGGL(pack_params, dim3((count + 255) / 256), dim3(256), 0, n->stream, dev,
                       static_cast<float *>(packed->get()), pk, static_cast<int>(count));
    CTAS_HIP_TRY(hipGetLastError());
    CTAS_HIP_TRY(hipStreamSynchronize(n->stream));
    CTAS_HIP_TRY(hipMemcpy(host, packed->get(), count * 4, hipMemcpyDeviceToHost));
    packed->done();
    return CTAS_OK;
  }
  CTAS_HIP_TRY(hipStreamSynchronize(n->stream));
  size_t at = 0;
  for (const auto &p : n->prm) {
    if (to_host)
      CTAS_HIP_TRY(hipMemcpy(host + at, dev + p.off, p.n * 4, hipMemcpyDeviceToHost));
    else
      CTAS_HIP_TRY(hipMemcpy(const_cast<float *>(dev) + p.off, host + at, p.n * 4, hipMemcpyHostToDevice));
    at += p.n;
  }
  return CTAS_OK;
}

extern "C" int ctas_cnn_get_params(ctas_cnn *n, float *params) {
  if (!n || !params) return fail(CTAS_E_ARG, "null argument");
  return copy_params(n, params, n->p, true);
}

extern "C" int ctas_cnn_get_grads(ctas_cnn *n, float *grads) {
  if (!n || !grads) return fail(CTAS_E_ARG, "null argument");
  return copy_params(n, grads, n->g, true);
}

extern "C" int ctas_cnn_set_params(ctas_cnn *n, const float *params) {
  if (!n || !params) return fail(CTAS_E_ARG, "null argument");
  if (int rc = copy_params(n, const_cast<float *>(params), n->p, false)) return rc;
  hipLaunchKernelGGL(to_bf16, dim3((n->nparam + 255) / 256), dim3(256), 0, n->stream, n->p, n->p16,
                     static_cast<int>(n->nparam));
  CTAS_HIP_TRY(hipStreamSynchronize(n->stream));
  return CTAS_OK;
}

// The _dev calls read inputs made ready on `stream` (nullptr: the null
// stream), run on the network's own stream and return when their results
// are complete.
extern "C" int ctas_cnn_forward_dev(ctas_cnn *n, const uint16_t *d_x, int B, float *d_out, void *stream) {
  if (!n || !d_x || !d_out || B <= 0) return fail(CTAS_E_ARG, "bad arguments");
  if (int rc = stream_wait(n->stream, static_cast<hipStream_t>(stream))) return rc;
  if (int rc = ensure_batch(n, B)) return rc;
  if (int rc = forward(n, d_x, B, false, n->out)) return rc;
  CTAS_HIP_TRY(hipMemcpyAsync(d_out, n->out, sizeof(float) * kOut * B, hipMemcpyDeviceToDevice, n->stream));
  CTAS_HIP_TRY(hipStreamSynchronize(n->stream));
  return CTAS_OK;
}

// Loss and parameter gradients of a batch (no update); loss on the host.
extern "C" int ctas_cnn_gradients_dev(ctas_cnn *n, const uint16_t *d_x, const float *d_target, int B, float *loss,
                                      void *stream) {
  if (!n || !d_x || !d_target || B <= 0) return fail(CTAS_E_ARG, "bad arguments");
  if (int rc = stream_wait(n->stream, static_cast<hipStream_t>(stream))) return rc;
  if (int rc = ensure_batch(n, B)) return rc;
  if (int rc = forward(n, d_x, B, true, n->out)) return rc;
  hipLaunchKernelGGL(loss_kernel, dim3(1), dim3(256), 0, n->stream, n->out, d_target, n->h1, W16(n, 10), n->gout,
                     n->host ? n->host + 2 : n->loss, G32(n, 10), G32(n, 11), n->gh1, G32(n, 9), B);
  if (int rc = backward(n, d_x, B)) return rc;
  CTAS_HIP_TRY(hipStreamSynchronize(n->stream));
  if (loss && n->host) *loss = n->host[2];
  else if (loss) CTAS_HIP_TRY(hipMemcpy(loss, n->loss, sizeof(float), hipMemcpyDeviceToHost));
  return CTAS_OK;
}

// Gradients + one Adam step (beta 0.9 / 0.999, eps 1e-8) at rate lr, the
// gradient scaled down to global norm clip_norm when it is larger (no
// clipping for clip_norm <= 0); grad_norm (optional) receives the norm
// before clipping.
extern "C" int ctas_cnn_train_step_dev(ctas_cnn *n, const uint16_t *d_x, const float *d_target, int B, float lr,
                                       float clip_norm, float *loss, float *grad_norm, void *stream) {
  if (int rc = ctas_cnn_gradients_dev(n, d_x, d_target, B, loss, stream)) return rc;
  ++n->step;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.0f - std::pow(b1, static_cast<float>(n->step));
  const float c2 = 1.0f - std::pow(b2, static_cast<float>(n->step));
  const int np = static_cast<int>(n->nparam);
  hipLaunchKernelGGL(sumsq_kernel, dim3(kNormBlocks), dim3(256), 0, n->stream, n->g, np, n->norm);
  hipLaunchKernelGGL(clip_factor_kernel, dim3(1), dim3(256), 0, n->stream, n->norm, clip_norm, n->norm + kNormBlocks);
  hipLaunchKernelGGL(adam_kernel, dim3((n->nparam + 255) / 256), dim3(256), 0, n->stream, n->p, n->p16, n->g, n->m,
                     n->v, np, lr, b1, b2, c1, c2, 1e-8f, n->norm + kNormBlocks);
  if (grad_norm) {
    CTAS_HIP_TRY(hipMemcpyAsync(grad_norm, n->norm + kNormBlocks + 1, sizeof(float), hipMemcpyDeviceToHost, n->stream));
  }
  CTAS_HIP_TRY(hipStreamSynchronize(n->stream));
  return CTAS_OK;
}

// Features of one sinogram [N][w] (device, transmission) into d_x
// [2][180][256]; work on `stream` (the caller's data must be ready there).
extern "C" int ctas_cnn_features_dev(const float *d_sino, int N, int w, uint16_t *d_x, void *stream) {
  if (!d_sino || !d_x || N < 1 || w < 2) return fail(CTAS_E_ARG, "bad arguments");
  hipStream_t s = static_cast<hipStream_t>(stream);
  float *tmp = nullptr;
  if (hipMalloc(&tmp, sizeof(float) * kFeatA * kFeatW) != hipSuccess) return fail(CTAS_E_NOMEM, "allocation failed");
  hipError_t e = launch_features(d_sino, N, w, tmp, d_x, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  (void)hipFree(tmp);
  if (e != hipSuccess) return fail(CTAS_E_DEVICE, std::string("features: ") + hipGetErrorString(e));
  return CTAS_OK;
}

extern "C" int ctas_cnn_save(const ctas_cnn *n, const char *path) {
  if (!n || !path) return fail(CTAS_E_ARG, "null argument");
  int c = 0;
  ctas_cnn_num_params(n, &c);
  std::vector<float> h(c);
  if (int rc = ctas_cnn_get_params(const_cast<ctas_cnn *>(n), h.data())) return rc;
  std::ofstream f(path, std::ios::binary);
  if (!f) return fail(CTAS_E_ARG, std::string("cannot write ") + path);
  const char magic[8] = {'C', 'T', 'A', 'S', 'C', 'N', 'N', '1'};
  f.write(magic, 8);
  f.write(reinterpret_cast<const char *>(&c), 4);
  f.write(reinterpret_cast<const char *>(h.data()), static_cast<std::streamsize>(h.size() * 4));
  return CTAS_OK;
}

extern "C" int ctas_cnn_load(ctas_cnn *n, const char *path) {
  if (!n || !path) return fail(CTAS_E_ARG, "null argument");
  std::ifstream f(path, std::ios::binary);
  if (!f) return fail(CTAS_E_ARG, std::string("cannot read ") + path);
  char magic[8];
  int c = 0, want = 0;
  f.read(magic, 8);
  f.read(reinterpret_cast<char *>(&c), 4);
  ctas_cnn_num_params(n, &want);
  if (!f || std::memcmp(magic, "CTASCNN1", 8) != 0 || c != want)
    return fail(CTAS_E_ARG, std::string("not a CNN weight file of this network: ") + path);
  std::vector<float> h(c);
  f.read(reinterpret_cast<char *>(h.data()), static_cast<std::streamsize>(h.size() * 4));
  if (!f) return fail(CTAS_E_ARG, std::string("truncated weight file ") + path);
  return ctas_cnn_set_params(n, h.data());
}

// ---- engine-made training samples ------------------------------------------
namespace {

uint64_t mix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}
double unit01(uint64_t h) { return (static_cast<double>(h >> 11) + 0.5) * (1.0 / 9007199254740992.0); }

constexpr int kBigEll = 20, kDots = 40;

}  // namespace

// Sample `index` of the stream `seed`: width w in {1024, 1280, ..., 4096},
// angles N in {900, 1200, 1500, 1800} over 180 degrees, centre offset c
// uniform in [-20, 20] px, photons per ray N0 log-uniform in [1e4, 1e6],
// 20 random ellipses (ctas_phantom_ellipses, semi-axes scaled by w/512)
// plus 40 dense inclusions (semi-axes 1-3 px, 0.03-0.09 per px) whose sharp
// edges give the average-gradient score its minimum at the true centre.
// ell receives (20 + 40) * 6 doubles; returns the ellipse count.
extern "C" int ctas_axis_sample(uint64_t seed, uint64_t index, int *w, int *N, double *c, double *N0, double *ell,
                                int *n_ell) {
  if (!w || !N || !c || !N0 || !ell || !n_ell) return fail(CTAS_E_ARG, "null argument");
  uint64_t st = mix64(seed ^ mix64(index + 0x51ed2701ull));
  auto next = [&]() {
    st = mix64(st);
    return unit01(st);
  };
  *w = 1024 + 256 * std::min(12, static_cast<int>(next() * 13));
  *N = 900 + 300 * std::min(3, static_cast<int>(next() * 4));
  *c = -20.0 + 40.0 * next();
  *N0 = std::pow(10.0, 4.0 + 2.0 * next());
  const uint64_t eseed = mix64(st ^ 0xe11a5e5ull);
  if (int rc = ctas_phantom_ellipses(kBigEll, *w, *w / 512.0, eseed, ell)) return rc;
  const double R = 0.5 * *w;
  for (int k = 0; k < kDots; ++k) {
    double *E = ell + 6 * (kBigEll + k);
    const double rr = 0.8 * R * std::sqrt(next());
    const double ang = 2.0 * M_PI * next();
    E[0] = rr * std::cos(ang);
    E[1] = rr * std::sin(ang);
    E[2] = 1.0 + 2.0 * next();
    E[3] = 1.0 + 2.0 * next();
    E[4] = M_PI * next();
    E[5] = 0.03 + 0.06 * next();
  }
  *n_ell = kBigEll + kDots;
  return CTAS_OK;
}

// Network input and targets of samples first .. first+B-1 of `seed`:
// d_x [B][2][180][256] bf16, d_target [B][2] = {offset in downsampled bins,
// tolerance (1 px) in bins}; offsets_px (host, optional) receives the true
// offsets and widths_px the widths. The sinograms are projected on the GPU
// (ctas_phantom_sino_dev geometry) one at a time into a scratch buffer.
extern "C" int ctas_cnn_make_batch(uint64_t seed, uint64_t first, int B, uint16_t *d_x, float *d_target,
                                   float *offsets_px, int *widths_px, void *stream) {
  if (!d_x || !d_target || B <= 0) return fail(CTAS_E_ARG, "bad arguments");
  hipStream_t s = static_cast<hipStream_t>(stream);
  constexpr int kMaxEll = kBigEll + kDots;
  float *d_sino = nullptr, *d_tmp = nullptr;
  double *d_ell = nullptr;
  const size_t max_sino = static_cast<size_t>(4096) * 1800;
  int rc = CTAS_OK;
  if (hipMalloc(&d_sino, sizeof(float) * max_sino) != hipSuccess ||
      hipMalloc(&d_tmp, sizeof(float) * kFeatA * kFeatW) != hipSuccess ||
      hipMalloc(&d_ell, sizeof(double) * 6 * kMaxEll * static_cast<size_t>(B)) != hipSuccess)
    rc = fail(CTAS_E_NOMEM, "allocation failed");
  std::vector<double> ell(static_cast<size_t>(6) * kMaxEll * B);
  std::vector<float> tgt(2 * static_cast<size_t>(B));
  std::vector<int> ws(B), Ns(B), ne(B);
  std::vector<double> cs(B), n0s(B);
  for (int b = 0; b < B && !rc; ++b)
    rc = ctas_axis_sample(seed, first + b, &ws[b], &Ns[b], &cs[b], &n0s[b], ell.data() + 6 * kMaxEll * b, &ne[b]);
  if (!rc && hipMemcpyAsync(d_ell, ell.data(), sizeof(double) * ell.size(), hipMemcpyHostToDevice, s) != hipSuccess)
    rc = fail(CTAS_E_DEVICE, "copy failed");
  for (int b = 0; b < B && !rc; ++b) {
    const double bin = ws[b] / static_cast<double>(kFeatW);
    tgt[2 * b] = static_cast<float>(cs[b] / bin);
    tgt[2 * b + 1] = static_cast<float>(1.0 / bin);
    if (offsets_px) offsets_px[b] = static_cast<float>(cs[b]);
    if (widths_px) widths_px[b] = ws[b];
    const uint64_t nseed = mix64(seed * 0x9E3779B97F4A7C15ull + first + b);
    if (launch_phantom(Ns[b], ws[b], cs[b], ne[b], d_ell + 6 * kMaxEll * b, n0s[b], nseed, nullptr, d_sino, s) !=
            hipSuccess ||
        launch_features(d_sino, Ns[b], ws[b], d_tmp, d_x + static_cast<size_t>(b) * 2 * kFeatA * kFeatW, s) !=
            hipSuccess)
      rc = fail(CTAS_E_DEVICE, "sample generation launch failed");
  }
  if (!rc && hipMemcpyAsync(d_target, tgt.data(), sizeof(float) * tgt.size(), hipMemcpyHostToDevice, s) != hipSuccess)
    rc = fail(CTAS_E_DEVICE, "copy failed");
  if (hipStreamSynchronize(s) != hipSuccess && !rc) rc = fail(CTAS_E_DEVICE, "sample generation failed");
  if (d_sino) (void)hipFree(d_sino);
  if (d_tmp) (void)hipFree(d_tmp);
  if (d_ell) (void)hipFree(d_ell);
  return rc;
}

// Offset (full-resolution px) and confidence of one device sinogram.
extern "C" int ctas_cnn_predict_dev(ctas_cnn *n, const float *d_sino, int N, int w, float *offset,
                                    float *confidence, void *stream) {
  if (!n || !d_sino || !offset || !confidence || N < 1 || w < 2) return fail(CTAS_E_ARG, "bad arguments");
  if (int rc = stream_wait(n->stream, static_cast<hipStream_t>(stream))) return rc;
  if (int rc = ensure_batch(n, 1)) return rc;
  if (!n->xin && alloc(reinterpret_cast<void **>(&n->xin), 2 * kFeatA * kFeatW * 2)) return CTAS_E_NOMEM;
  CTAS_HIP_TRY(launch_features(d_sino, N, w, n->ftmp, n->xin, n->stream));
  // the last kernel writes to the host: with a copy of the eight bytes a
  // prediction takes 99 us, so 82
  if (int rc = forward(n, n->xin, 1, false, n->host ? n->host : n->out)) return rc;
  float o[2];
  if (!n->host) CTAS_HIP_TRY(hipMemcpyAsync(o, n->out, sizeof(o), hipMemcpyDeviceToHost, n->stream));
  CTAS_HIP_TRY(hipStreamSynchronize(n->stream));
  if (n->host) std::memcpy(o, n->host, sizeof(o));
  *offset = o[0] * static_cast<float>(w) / kFeatW;
  *confidence = 1.0f / (1.0f + std::exp(-o[1]));
  return CTAS_OK;
}

// Same for a host sinogram.
extern "C" int ctas_cnn_predict(ctas_cnn *n, const float *sino, int N, int w, float *offset, float *confidence) {
  if (!n || !sino || !offset || !confidence || N < 1 || w < 2) return fail(CTAS_E_ARG, "bad arguments");
  float *d_s = nullptr;
  if (hipMalloc(&d_s, sizeof(float) * N * w) != hipSuccess) return fail(CTAS_E_NOMEM, "allocation failed");
  int rc = CTAS_OK;
  if (hipMemcpy(d_s, sino, sizeof(float) * N * w, hipMemcpyHostToDevice) != hipSuccess)
    rc = fail(CTAS_E_DEVICE, "copy failed");
  if (!rc) rc = ctas_cnn_predict_dev(n, d_s, N, w, offset, confidence, nullptr);
  (void)hipFree(d_s);
  return rc;
}

// Sweep of trial centres offsets -half_range + k*step (k = 0 .. K-1) on the
// device sinogram d_sino of handle h's shape (AverageGradient canon: ABS,
// RAMP); result = the offset of the lowest score (first on ties). With a
// network whose confidence reaches min_confidence, only a window of 3 grid
// points around its estimate is scored, widened by one point on the side of
// its lowest score while that is at an edge (and not the grid's end); past
// kMaxWindow points the remaining grid is scored too. info
// (optional, 4 ints): trials scored, 1 if the whole grid was swept,
// network estimate (milli-px), confidence (per mille).
constexpr int kMaxWindow = 21;

namespace {

// The sweep of ctas_axis_find on a device sinogram: with `windowed`, a
// window of 3 grid points around `start` (px), widened one point at a time
// towards a lower edge score until its minimum is interior, the whole grid
// past kMaxWindow points; otherwise the whole grid. est and conf only go to
// info.
// Argument checks and the filter of the sinogram on the handle's stream
// (after the work already queued on the null stream, which the caller's
// NullStreamJoin orders).
int axis_prepare(ctas_fbp *h, const float *d_sino, float half_range, float step, float *offset) {
  if (!h || !d_sino || !offset || !(step > 0) || !(half_range >= 0)) return fail(CTAS_E_ARG, "bad arguments");
  const int K = static_cast<int>(std::floor(2.0 * half_range / step + 0.5)) + 1;
  if (K > 4096) return fail(CTAS_E_ARG, "too many trial centres");
  if (std::ceil(half_range) >= 0.5f * h->w) return fail(CTAS_E_CENTER, "trial centres beyond half the width");
  return ctas_fbp_prepare_dev(h, d_sino, 1, h->stream);
}

// The search itself, on the filtered sinogram axis_prepare left.
int axis_search(ctas_fbp *h, float half_range, float step, bool windowed, float start, float est, float conf,
                float *offset, int *info) {
  const int w = h->w;
  const int K = static_cast<int>(std::floor(2.0 * half_range / step + 0.5)) + 1;
  const float cent = static_cast<float>(0.5 * (w - 1));
  auto grid = [&](int k) { return static_cast<float>(-static_cast<double>(half_range) + k * static_cast<double>(step)); };
  std::vector<float> sc(K, 0.0f);
  std::vector<char> have(K, 0);
  int trials = 0;
  auto eval = [&](int lo, int hi) -> int {
    std::vector<float> ax;
    std::vector<int> ks;
    for (int k = lo; k <= hi; ++k)
      if (!have[k]) {
        ax.push_back(cent + grid(k));
        ks.push_back(k);
      }
    if (ax.empty()) return CTAS_OK;
    std::vector<float> v(ax.size());
    if (int rc = ctas_axis_scores(h, ax.data(), static_cast<int>(ax.size()), v.data())) return rc;
    for (size_t i = 0; i < ks.size(); ++i) {
      sc[ks[i]] = v[i];
      have[ks[i]] = 1;
    }
    trials += static_cast<int>(ks.size());
    return CTAS_OK;
  };
  auto argmin = [&](int lo, int hi) {
    int m = lo;
    for (int k = lo + 1; k <= hi; ++k)
      if (sc[k] < sc[m]) m = k;
    return m;
  };
  int swept = 1, km = 0;
  if (windowed) {
    swept = 0;
    const int k0 = std::max(0, std::min(K - 1, static_cast<int>(std::lround((start + half_range) / step))));
    int lo = std::max(0, k0 - 1), hi = std::min(K - 1, k0 + 1);
    if (int rc = eval(lo, hi)) return rc;
    for (;;) {
      km = argmin(lo, hi);
      if (hi - lo + 1 > kMaxWindow) {
        swept = 1;
        break;
      }
      if (km == lo && lo > 0) {
        --lo;
      } else if (km == hi && hi < K - 1) {
        ++hi;
      } else {
        break;
      }
      if (int rc = eval(lo, hi)) return rc;
    }
  }
  if (swept) {
    if (int rc = eval(0, K - 1)) return rc;
    km = argmin(0, K - 1);
  }
  *offset = grid(km);
  if (info) {
    info[0] = trials;
    info[1] = swept;
    info[2] = static_cast<int>(std::lround(est * 1000.0f));
    info[3] = static_cast<int>(std::lround(conf * 1000.0f));
  }
  return CTAS_OK;
}

}  // namespace

extern "C" int ctas_axis_find(ctas_fbp *h, ctas_cnn *net, const float *d_sino, float half_range, float step,
                              float min_confidence, float *offset, int *info) {
  if (!h) return fail(CTAS_E_ARG, "bad arguments");
  // filtering on the handle's stream, the network on its own stream, both
  // after the work already queued on the null stream
  NullStreamJoin join(h->stream, nullptr);
  if (join.rc) return join.rc;
  if (int rc = axis_prepare(h, d_sino, half_range, step, offset)) return rc;
  float est = 0.0f, conf = 0.0f;
  if (net) {
    if (int rc = ctas_cnn_predict_dev(net, d_sino, h->N, h->w, &est, &conf, nullptr)) return rc;
  }
  return axis_search(h, half_range, step, net && conf >= min_confidence, est, est, conf, offset, info);
}

extern "C" int ctas_axis_find_from(ctas_fbp *h, const float *d_sino, float half_range, float step, float start,
                                   float *offset, int *info) {
  if (!h) return fail(CTAS_E_ARG, "bad arguments");
  NullStreamJoin join(h->stream, nullptr);
  if (join.rc) return join.rc;
  if (int rc = axis_prepare(h, d_sino, half_range, step, offset)) return rc;
  return axis_search(h, half_range, step, true, start, start, 1.0f, offset, info);
}

// bf16 GEMM of the network's kernel on plain row-major operands:
// C[M][N] (fp32) = A[M][K] x B[K][N] (bf16). Exposed for verification of the
// matrix-core operand layout.
extern "C" int ctas_cnn_gemm_dev(const uint16_t *d_a, const uint16_t *d_b, float *d_c, int M, int N, int K,
                                 void *stream) {
  if (!d_a || !d_b || !d_c || M <= 0 || N <= 0 || K <= 0) return fail(CTAS_E_ARG, "bad arguments");
  hipStream_t s = static_cast<hipStream_t>(stream);
  CTAS_HIP_TRY(gemm(DenseA{d_a, K}, ActBT{d_b, N}, StoreDX{d_c, 1, 1, N}, M, N, K, s));  // on the caller's stream
  CTAS_HIP_TRY(hipStreamSynchronize(s));
  return CTAS_OK;
}

// CNN-fronted axis search: the network's estimate replaces the sweep of
// raxis algorithm 1 (lct.cpp:1183-1205); the score is evaluated at the
// estimate (rounded to 0.25 px) and +-4 px around it in one batch, and
// improveMe (lct.cpp:1108-1129) refines from that bracket with the same
// tolerance (0.25 px). Falls back to ctas_raxis (algorithm 1) when the
// confidence is below min_confidence, the estimate is outside maxDev, or
// the centre of the bracket is not its lowest score; the argument checks
// and their errors are those of ctas_raxis.
extern "C" int ctas_raxis_cnn(ctas_cnn *n, const float *sino, int N, int w, float anarc, float maxDev,
                              float min_confidence, float *result, int *used_sweep) {
  if (!n || !sino || !result) return fail(CTAS_E_ARG, "null argument");
  if (used_sweep) *used_sweep = 0;
  auto sweep = [&]() {
    if (used_sweep) *used_sweep = 1;
    return ctas_raxis(sino, N, w, anarc, maxDev, 1, result);
  };
  const float arc = N > 1 ? arc_rad(anarc, N) : 0.0f;
  if (N < 3 || w < 3 || std::fabs(arc) < static_cast<float>(M_PI) || maxDev < 0 || maxDev > 0.25f) return sweep();
  float off = 0.0f, conf = 0.0f;
  if (int rc = ctas_cnn_predict(n, sino, N, w, &off, &conf)) return rc;
  const float mid = static_cast<float>(0.5 * (w - 1));
  const float est_px = std::round(off * 4.0f) / 4.0f;
  if (!(conf >= min_confidence) || std::fabs(est_px) + 4.0f > maxDev * w) return sweep();
  ctas_fbp *h = nullptr;
  if (int rc = ctas_fbp_create(&h, w, N, CTAS_CONTRAST_ABS, CTAS_FILTER_RAMP, 0.0f, anarc, 0)) return rc;
  std::unique_ptr<ctas_fbp, int (*)(ctas_fbp *)> guard(h, ctas_fbp_destroy);
  std::vector<float> copy(sino, sino + static_cast<size_t>(N) * w);
  if (int rc = ctas_fbp_sino(h, copy.data())) return rc;
  const std::vector<float> offsets = {est_px - 4.0f, est_px, est_px + 4.0f};
  std::vector<float> scores(3);
  const float ax[3] = {mid + offsets[0], mid + offsets[1], mid + offsets[2]};
  if (int rc = ctas_axis_scores(h, ax, 3, scores.data())) return rc;
  if (!(scores[1] < scores[0] && scores[1] < scores[2])) {
    guard.reset();
    return sweep();
  }
  int rc = CTAS_OK;
  auto score_at = [&](float x) -> float {
    float axis = mid + x, v = 0.0f;
    if (!rc) rc = ctas_axis_scores(h, &axis, 1, &v);
    return v;
  };
  const float best = improve_me(0.25f, offsets, scores, 1, 1, score_at, &rc);
  if (rc) return rc;
  *result = mid + best;
  return CTAS_OK;
}
