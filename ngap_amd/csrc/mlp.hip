// Frontier-size predictor: a 264 -> 64 -> 64 -> 1 ReLU MLP in FP32, trained
// and evaluated with these kernels.  It predicts log(1 + items) of one
// (group, 4 KiB window) work item from the window's 256-bin byte histogram and
// 8 statistics of the group's automaton; the batched scheduler uses the
// prediction only to size and order work items.  No counterpart in the
// reference.
//
// Parameter layout (floats): W1[264][64], b1[64], W2[64][64], b2[64], W3[64],
// b3[1].  Features of sample n are either a dense row X[n][264] or, for
// inference over many (group, window) pairs, the concatenation of
// hist[window][256] and stats[group][8].
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/ngap_amd.h"
#include "c_guard.h"

void ngap_set_last_error_internal(const std::string &m) noexcept;

namespace {

constexpr int kIn = 264, kHid = 64, kHist = 256;
constexpr int kW1 = 0, kB1 = kW1 + kIn * kHid, kW2 = kB1 + kHid, kB2 = kW2 + kHid * kHid,
              kW3 = kB2 + kHid, kB3 = kW3 + kHid, kParams = kB3 + 1;

int fail(int code, const std::string &m) {
  ngap_set_last_error_internal(m);
  return code;
}
#define MLP_TRY(expr)                                                            \
  do {                                                                           \
    hipError_t _e = (expr);                                                      \
    if (_e != hipSuccess)                                                        \
      return fail(_e == hipErrorOutOfMemory ? NGAP_ERR_OOM : NGAP_ERR_DEVICE,    \
                  std::string(#expr) + ": " + hipGetErrorString(_e));            \
  } while (0)

// The products run on the FP32 matrix cores (v_mfma_f32_16x16x4: FP32 inputs
// and accumulation).  Each wave computes C = A B with the features as rows
// and the samples as columns: lane l holds sample l % 16 and, with q = l / 16,
// features 4 q .. 4 q + 3 of a 16-feature tile, so a layer's output is the
// next layer's B operand after one LDS exchange and the last layer is a dot
// product over a lane's registers.  Step (j, e) of a product takes the four
// inputs 16 j + 4 q + e (q = 0 .. 3): a lane's inputs of four steps are one
// 16-byte load.  Every path sums in this order, the histogram part and the
// statistics part of the first layer apart (with b1 in the latter), so a
// prediction has the same bits whichever path computes it.
typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f4 mfma(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4 load4(const float *p) { return *reinterpret_cast<const f4 *>(p); }
__device__ __forceinline__ void store4(float *p, f4 v) { *reinterpret_cast<f4 *>(p) = v; }
__device__ __forceinline__ f4 relu(f4 v) {
#pragma unroll
  for (int r = 0; r < 4; r++) v[r] = fmaxf(v[r], 0.f);
  return v;
}

// Histogram part of the first layer (unrolled by four: see k_gradient): features 16 ft .. 16 ft + 15 of the
// lane's sample, whose inputs are at x.
__device__ __forceinline__ f4 hist_part(const float *P, const float *x, int ft) {
  const int c = threadIdx.x % 16, q = threadIdx.x % 64 / 16;
  const float *W = P + kW1 + 16 * ft + c;
  f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int j = 0; j < kHist / 16; j++) {
    const int k = 16 * j + 4 * q;
    const f4 v = load4(x + k);
#pragma unroll
    for (int e = 0; e < 4; e++) acc = mfma(W[(k + e) * kHid], v[e], acc);
  }
  return acc;
}

// Statistics part (8 inputs) plus b1.
__device__ __forceinline__ f4 stats_part(const float *P, const float *x, int ft) {
  const int c = threadIdx.x % 16, q = threadIdx.x % 64 / 16;
  const float *W = P + kW1 + 16 * ft + c;
  f4 acc = load4(P + kB1 + 16 * ft + 4 * q);
#pragma unroll
  for (int e = 0; e < 2; e++)
    acc = mfma(W[(kHist + 2 * q + e) * kHid], x[2 * q + e], acc);
  return acc;
}

// Tiles of kTile samples, one workgroup of 8 waves: wave w owns the samples
// 16 (w / 4) .. + 15 and the features 16 (w % 4) .. + 15 of every layer.
// LDS rows are padded so that four rows 16 words apart fill the 64 banks.
constexpr int kTile = 32, kThreads = 16 * kTile, kHalves = kTile / 16;
constexpr int kXs = kIn + 8, kHs = kHid + 16;

// x[kTile][kXs] = the features of samples [s0, s0 + kTile) of X (rows idx[s]
// when given), zero past n and past kIn.
__device__ __forceinline__ void load_tile(float *x, const float *X, const uint32_t *idx,
                                          uint64_t n, uint64_t s0) {
  const f4 zero = {0.f, 0.f, 0.f, 0.f};
  for (int k = threadIdx.x; k < kTile * (kXs / 4); k += kThreads) {
    const int s = k / (kXs / 4), i = k % (kXs / 4) * 4;
    const uint64_t ns = s0 + s;
    f4 v = zero;
    if (ns < n && i < kIn) v = load4(X + (idx ? (uint64_t)idx[ns] : ns) * kIn + i);
    store4(x + s * kXs + i, v);
  }
}

// Second layer before its ReLU: features 16 ft .. of the lane's sample, whose
// first-layer outputs are at h.
__device__ __forceinline__ f4 layer2(const float *P, const float *h, int ft) {
  const int c = threadIdx.x % 16, q = threadIdx.x % 64 / 16;
  const float *W = P + kW2 + 16 * ft + c;
  f4 acc = load4(P + kB2 + 16 * ft + 4 * q);
#pragma unroll
  for (int j = 0; j < kHid / 16; j++) {
    const int k = 16 * j + 4 * q;
    const f4 v = load4(h + k);
#pragma unroll
    for (int e = 0; e < 4; e++) acc = mfma(W[(k + e) * kHid], v[e], acc);
  }
  return acc;
}

// A lane's share of the last layer.
__device__ __forceinline__ float dot3(f4 w3, f4 h2) {
  float p = 0.f;
#pragma unroll
  for (int r = 0; r < 4; r++) p = fmaf(h2[r], w3[r], p);
  return p;
}

// Forward of one tile: first-layer outputs of the wave's part in h1 (and in
// LDS for every wave), second-layer ones in h2, the tile's predictions in
// y[kTile].  Ends with a barrier.
__device__ __forceinline__ void forward_tile(const float *P, const float *x, float *lh1,
                                             float *yp, float *y, f4 &h1, f4 &h2) {
  const int t = threadIdx.x, ft = t / 64 % 4, s = t / 256 * 16 + t % 16, q = t % 64 / 16;
  h1 = relu(hist_part(P, x + s * kXs, ft) + stats_part(P, x + s * kXs + kHist, ft));
  store4(lh1 + s * kHs + 16 * ft + 4 * q, h1);
  __syncthreads();
  h2 = relu(layer2(P, lh1 + s * kHs, ft));
  yp[(ft * 4 + q) * kTile + s] = dot3(load4(P + kW3 + 16 * ft + 4 * q), h2);
  __syncthreads();
  if (t < kTile) {
    float part[4];
#pragma unroll
    for (int k = 0; k < 4; k++)
      part[k] = ((yp[k * kTile + t] + yp[(4 + k) * kTile + t]) + yp[(8 + k) * kTile + t]) +
                yp[(12 + k) * kTile + t];
    y[t] = ((part[0] + part[1]) + (part[2] + part[3])) + P[kB3];
  }
  __syncthreads();
}

// Predictions of n dense samples.
__global__ void __launch_bounds__(kThreads)
    k_forward(const float *P, const float *X, uint64_t n, float *Y) {
  __shared__ __align__(16) float x[kTile * kXs];
  __shared__ __align__(16) float lh1[kTile * kHs];
  __shared__ float yp[16 * kTile], y[kTile];
  for (uint64_t s0 = (uint64_t)blockIdx.x * kTile; s0 < n; s0 += (uint64_t)gridDim.x * kTile) {
    load_tile(x, X, nullptr, n, s0);
    __syncthreads();
    f4 h1, h2;
    forward_tile(P, x, lh1, yp, y, h1, h2);
    if (threadIdx.x < kTile && s0 + threadIdx.x < n) Y[s0 + threadIdx.x] = y[threadIdx.x];
  }
}

// First-layer parts for predict_pairs: a prediction's inputs are one of the
// windows' histograms and one of the groups' statistics, so the first layer
// is computed once per window and once per group, not once per pair (264 of
// the 329 multiply-adds per hidden unit and pair).  One wave per 16 rows and
// feature tile; blocks [0, wblocks) take windows, the others groups.
__global__ void __launch_bounds__(256)
    k_parts(const float *P, const float *hist, uint32_t num_windows, const float *stats,
            uint32_t num_groups, uint32_t wblocks, float *wpart, float *gpart,
            uint32_t *bad) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *bad = 0u;  // for k_pairs
  const bool win = blockIdx.x < wblocks;
  const uint32_t rows = win ? num_windows : num_groups;
  const uint32_t row = (blockIdx.x - (win ? 0 : wblocks)) * 16 + threadIdx.x % 16;
  const uint32_t at = row < rows ? row : rows - 1;  // a valid row for the idle lanes
  const int ft = threadIdx.x / 64, q = threadIdx.x % 64 / 16;
  const f4 v = win ? hist_part(P, hist + (uint64_t)at * kHist, ft)
                   : stats_part(P, stats + (uint64_t)at * 8, ft);
  if (row < rows) store4((win ? wpart : gpart) + (uint64_t)row * kHid + 16 * ft + 4 * q, v);
}

// Predictions of n (group, window) pairs from the parts.  A wave keeps W2 in
// 64 registers and takes 16 pairs per round: 64 matrix instructions, which
// bound the kernel, beside eight 16-byte loads, the sum and ReLU of the parts
// and the last layer.  2.1M pairs take 174 us (99 TFLOP/s of second-layer
// products, 154 being what a large FP32 product reaches here); with half of the
// products left out 102, with the gathers from 16 rows only 174, with the next
// round's parts loaded ahead (one workgroup fewer per CU) 198.  The whole first
// layer per pair on the vector units, as before: 2,656.  Pairs out of range set
// *bad.
__global__ void __launch_bounds__(256)
    k_pairs(const float *P, const float *wpart, const float *gpart, const uint2 *pairs,
            uint64_t n, uint32_t num_windows, uint32_t num_groups, float *Y, uint32_t *bad) {
  const int c = threadIdx.x % 16, q = threadIdx.x % 64 / 16;
  float w2[4][kHid / 4];
  f4 b2[4], w3[4];
#pragma unroll
  for (int ft = 0; ft < 4; ft++) {
#pragma unroll
    for (int i = 0; i < kHid / 4; i++)
      w2[ft][i] = P[kW2 + (16 * (i / 4) + 4 * q + i % 4) * kHid + 16 * ft + c];
    b2[ft] = load4(P + kB2 + 16 * ft + 4 * q);
    w3[ft] = load4(P + kW3 + 16 * ft + 4 * q);
  }
  const float b3 = P[kB3];
  const uint64_t waves = (uint64_t)gridDim.x * 4;
  uint64_t s0 = ((uint64_t)blockIdx.x * 4 + threadIdx.x / 64) * 16;
  uint2 pair = pairs[s0 + c < n ? s0 + c : 0];
  for (; s0 < n; s0 += waves * 16) {
    const uint64_t ahead = s0 + waves * 16 + c;
    const uint2 next = pairs[ahead < n ? ahead : 0];
    const bool ok = pair.x < num_groups && pair.y < num_windows;
    if (!ok) *bad = 1u;
    const float *gp = gpart + (uint64_t)(ok ? pair.x : 0) * kHid + 4 * q;
    const float *wp = wpart + (uint64_t)(ok ? pair.y : 0) * kHid + 4 * q;
    f4 h[4];
#pragma unroll
    for (int j = 0; j < 4; j++) h[j] = relu(load4(wp + 16 * j) + load4(gp + 16 * j));
    f4 acc[4];
#pragma unroll
    for (int ft = 0; ft < 4; ft++) acc[ft] = b2[ft];
#pragma unroll
    for (int i = 0; i < kHid / 4; i++)
#pragma unroll
      for (int ft = 0; ft < 4; ft++) acc[ft] = mfma(w2[ft][i], h[i / 4][i % 4], acc[ft]);
    float p = dot3(w3[0], relu(acc[0]));
#pragma unroll
    for (int ft = 1; ft < 4; ft++) p += dot3(w3[ft], relu(acc[ft]));
    p += __shfl_xor(p, 16, 64);
    p += __shfl_xor(p, 32, 64);
    if (q == 0 && s0 + c < n) Y[s0 + c] = p + b3;
    pair = next;
  }
}

// Gradient of the mean squared error: forward and backward in one kernel, so
// that no activation leaves the chip.  Each workgroup runs its tiles forward
// and backward and leaves its sums in G[block][kPart] (the loss after the
// gradient); k_reduce adds the workgroups' rows.  The weight gradients
// (samples as the summed dimension) stay in matrix accumulators over a
// workgroup's tiles: wave w owns output tiles (., w % 4) of dW1 (17 row
// tiles, every second one from w / 4) and of dW2.
constexpr int kPart = (kParams + 1 + 63) / 64 * 64;
constexpr int kMaxGradBlocks = 512;
constexpr int kRow1 = kXs / 16;  // row tiles of dW1 (the last one half padding)
constexpr int kTiles1 = (kRow1 + kHalves - 1) / kHalves, kTiles2 = 4 / kHalves;  // of a wave
constexpr size_t kGradLds = (size_t)(kTile * kXs + 3 * kTile * kHs + 18 * kTile) * 4;

__global__ void __launch_bounds__(kThreads)
    k_gradient(const float *P, const float *X, const float *T, const uint32_t *idx, uint64_t n,
               float *G) {
  extern __shared__ __align__(16) float lds[];
  float *x = lds;                  // [kTile][kXs]
  float *lh1 = x + kTile * kXs;    // [kTile][kHs]
  float *ld2 = lh1 + kTile * kHs;
  float *ld1 = ld2 + kTile * kHs;
  float *yp = ld1 + kTile * kHs;   // [16][kTile]
  float *y = yp + 16 * kTile;      // [kTile]
  float *dy = y + kTile;
  const int t = threadIdx.x, w = t / 64, c = t % 16, q = t % 64 / 16;
  const int ft = w % 4, half = w / 4, s = half * 16 + c;
  const f4 zero = {0.f, 0.f, 0.f, 0.f};
  const f4 w3 = load4(P + kW3 + 16 * ft + 4 * q);
  f4 gw1[kTiles1], gw2[kTiles2];
#pragma unroll
  for (int m = 0; m < kTiles1; m++) gw1[m] = zero;
#pragma unroll
  for (int m = 0; m < kTiles2; m++) gw2[m] = zero;
  f4 gw3 = zero, gb1 = zero, gb2 = zero;
  float gb3 = 0.f, loss = 0.f;
  const float scale = 2.0f / (float)n;
  for (uint64_t s0 = (uint64_t)blockIdx.x * kTile; s0 < n; s0 += (uint64_t)gridDim.x * kTile) {
    load_tile(x, X, idx, n, s0);
    __syncthreads();
    f4 h1, h2;
    forward_tile(P, x, lh1, yp, y, h1, h2);
    if (t < kTile) {
      const uint64_t ns = s0 + t;
      const float e = ns < n ? y[t] - T[idx ? idx[ns] : ns] : 0.f;
      dy[t] = e * scale;
      loss = fmaf(e, e, loss);
      gb3 += e * scale;
    }
    __syncthreads();
    // d2 = dy W3^T relu'(h2), d1 = d2 W2^T relu'(h1): each wave its part
    const float dys = dy[s];
    f4 d2;
#pragma unroll
    for (int r = 0; r < 4; r++) d2[r] = h2[r] > 0.f ? dys * w3[r] : 0.f;
    store4(ld2 + s * kHs + 16 * ft + 4 * q, d2);
    gw3 += h2 * dys;
    gb2 += d2;
    __syncthreads();
    f4 d1 = zero;
    const float *W = P + kW2 + (16 * ft + c) * kHid + 4 * q;
#pragma unroll
    for (int j = 0; j < kHid / 16; j++) {
      const f4 a = load4(W + 16 * j), b = load4(ld2 + s * kHs + 16 * j + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; e++) d1 = mfma(a[e], b[e], d1);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) d1[r] = h1[r] > 0.f ? d1[r] : 0.f;
    store4(ld1 + s * kHs + 16 * ft + 4 * q, d1);
    gb1 += d1;
    __syncthreads();
    // dW1 = X^T d1, dW2 = h1^T d2: step k takes samples 4 k .. 4 k + 3
    float b1[kTile / 4], b2[kTile / 4];
#pragma unroll
    for (int k = 0; k < kTile / 4; k++) {
      b1[k] = ld1[(4 * k + q) * kHs + 16 * ft + c];
      b2[k] = ld2[(4 * k + q) * kHs + 16 * ft + c];
    }
#pragma unroll
    for (int m = 0; m < kTiles1; m++) {
      const int row = kHalves * m + half;
      if (row < kRow1)  // wave-uniform
#pragma unroll
        for (int k = 0; k < kTile / 4; k++)
          gw1[m] = mfma(x[(4 * k + q) * kXs + 16 * row + c], b1[k], gw1[m]);
    }
#pragma unroll
    for (int m = 0; m < kTiles2; m++)
#pragma unroll
      for (int k = 0; k < kTile / 4; k++)
        gw2[m] = mfma(lh1[(4 * k + q) * kHs + 16 * (kHalves * m + half) + c], b2[k], gw2[m]);
    __syncthreads();  // the next tile overwrites x, lh1, ld1 and ld2
  }
  float *out = G + (uint64_t)blockIdx.x * kPart;
#pragma unroll
  for (int m = 0; m < kTiles1; m++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = 16 * (kHalves * m + half) + 4 * q + r;
      if (i < kIn) out[kW1 + i * kHid + 16 * ft + c] = gw1[m][r];
    }
#pragma unroll
  for (int m = 0; m < kTiles2; m++)
#pragma unroll
    for (int r = 0; r < 4; r++)
      out[kW2 + (16 * (kHalves * m + half) + 4 * q + r) * kHid + 16 * ft + c] = gw2[m][r];
  // sums over samples: a lane's sample column, then the two halves of the
  // tile (through lh1, free now: [half][3][kHid])
#pragma unroll
  for (int d = 1; d < 16; d <<= 1)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      gw3[r] += __shfl_xor(gw3[r], d, 64);
      gb1[r] += __shfl_xor(gb1[r], d, 64);
      gb2[r] += __shfl_xor(gb2[r], d, 64);
    }
  if (c == 0) {
    float *o = lh1 + half * 3 * kHid + 16 * ft + 4 * q;
    store4(o, gw3);
    store4(o + kHid, gb1);
    store4(o + 2 * kHid, gb2);
  }
  if (t < 64) {
#pragma unroll
    for (int d = 1; d < 32; d <<= 1) {
      loss += __shfl_xor(loss, d, 64);
      gb3 += __shfl_xor(gb3, d, 64);
    }
    if (t == 0) {
      out[kB3] = gb3;
      out[kParams] = loss;
    }
  }
  __syncthreads();
  if (t < kHid) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      float a = lh1[k * kHid + t];
#pragma unroll
      for (int h = 1; h < kHalves; h++) a += lh1[(3 * h + k) * kHid + t];
      out[(k == 0 ? kW3 : k == 1 ? kB1 : kB2) + t] = a;
    }
  }
}

struct Adam {
  float lr, b1, b2, eps, c1, c2;
};

// Adds the workgroups' rows (four waves take every fourth one each); then the
// gradient goes to `grad`, or, when that is null, into an Adam step on P.  The
// sum behind the parameters is the loss.
__global__ void __launch_bounds__(256)
    k_reduce(const float *G, int rows, float *grad, float *loss, float *P, float *M, float *V,
             Adam o) {
  __shared__ float part[4][64];
  const int i = blockIdx.x * 64 + threadIdx.x % 64, w = threadIdx.x / 64;
  float a = 0.f;
#pragma unroll 8
  for (int r = w; r < rows; r += 4) a += G[(uint64_t)r * kPart + i];
  part[w][threadIdx.x % 64] = a;
  __syncthreads();
  if (w != 0 || i > kParams) return;
  const float g = (part[0][threadIdx.x] + part[1][threadIdx.x]) +
                  (part[2][threadIdx.x] + part[3][threadIdx.x]);
  if (i == kParams) {
    *loss = g;
  } else if (grad) {
    grad[i] = g;
  } else {
    const float m = o.b1 * M[i] + (1.f - o.b1) * g;
    const float v = o.b2 * V[i] + (1.f - o.b2) * g * g;
    M[i] = m;
    V[i] = v;
    P[i] -= o.lr * (m / o.c1) / (sqrtf(v / o.c2) + o.eps);
  }
}

struct Buf {
  void *p = nullptr;
  size_t n = 0;
  ~Buf() { release(); }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  hipError_t reserve(size_t bytes) {
    if (bytes <= n && p) return hipSuccess;
    release();
    hipError_t e = hipMalloc(&p, bytes ? bytes : 8);
    if (e == hipSuccess) n = bytes ? bytes : 8;
    return e;
  }
  float *f() const { return reinterpret_cast<float *>(p); }
};

}  // namespace

// Samples that training keeps on the device while it runs, at most (15M), and
// that the model goes on holding afterwards, for the next training (254,000).
constexpr uint64_t kResident = 16ull << 30, kHeld = 256ull << 20;

struct ngap_mlp {
  int device = 0;
  Buf P, G, M, V, loss;
  Buf X, T, Y, hist, stats, pairs, parts, idx;
  int step = 0;
};

namespace {

uint32_t blocks_for(uint64_t n, uint64_t per_block, uint64_t most) {
  return (uint32_t)std::min<uint64_t>((n + per_block - 1) / per_block, most);
}

// k_gradient's workgroups over n samples, and what their sums take
uint32_t grad_blocks(uint64_t n) { return blocks_for(n, kTile, kMaxGradBlocks); }
size_t grad_bytes(uint64_t n) { return (size_t)grad_blocks(n) * kPart * 4; }

int load_batch(ngap_mlp *m, const float *x, const float *t, uint64_t n) {
  MLP_TRY(m->X.reserve(n * kIn * 4));
  MLP_TRY(hipMemcpy(m->X.p, x, n * kIn * 4, hipMemcpyHostToDevice));
  if (t) {
    MLP_TRY(m->T.reserve(n * 4));
    MLP_TRY(hipMemcpy(m->T.p, t, n * 4, hipMemcpyHostToDevice));
  }
  return NGAP_OK;
}

// Gradient over n resident samples (rows idx[0, n) when given), into grad, or
// as an Adam step when grad is null; the loss sum goes to *loss (device).
int grad_on_device(ngap_mlp *m, const uint32_t *idx, uint64_t n, float *grad, float *loss,
                   const Adam &o) {
  const uint32_t blocks = grad_blocks(n);
  MLP_TRY(m->G.reserve(grad_bytes(n)));
  hipLaunchKernelGGL(k_gradient, dim3(blocks), dim3(kThreads), kGradLds, 0, m->P.f(), m->X.f(),
                     m->T.f(), idx, n, m->G.f());
  MLP_TRY(hipGetLastError());
  hipLaunchKernelGGL(k_reduce, dim3(kPart / 64), dim3(256), 0, 0, m->G.f(), (int)blocks, grad,
                     loss, m->P.f(), m->M.f(), m->V.f(), o);
  MLP_TRY(hipGetLastError());
  return NGAP_OK;
}

}  // namespace

extern "C" {

int ngap_mlp_create(int32_t device, uint64_t seed, ngap_mlp **out) {
  return ngapamd::c_guard([&]() -> int {
    if (!out) return fail(NGAP_ERR_INVALID, "NULL argument");
    *out = nullptr;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count == 0)
      return fail(NGAP_ERR_DEVICE, "no HIP device available");
    MLP_TRY(hipSetDevice(device));
    MLP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(k_gradient),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)kGradLds));
    ngap_mlp *m = new ngap_mlp();
    m->device = device;
    std::vector<float> p(kParams, 0.f);
    // He-uniform initialisation from a splitmix64 stream
    uint64_t z = seed + 0x9E3779B97F4A7C15ull;
    auto next = [&]() {
      z += 0x9E3779B97F4A7C15ull;
      uint64_t x = z;
      x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
      x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
      x ^= x >> 31;
      return (double)(x >> 11) / 9007199254740992.0;
    };
    auto fill = [&](int off, int cnt, int fan_in) {
      const double a = std::sqrt(6.0 / fan_in);
      for (int i = 0; i < cnt; i++) p[off + i] = (float)((2 * next() - 1) * a);
    };
    fill(kW1, kIn * kHid, kIn);
    fill(kW2, kHid * kHid, kHid);
    fill(kW3, kHid, kHid);
    int rc = NGAP_OK;
    if (m->P.reserve(kParams * 4) || m->M.reserve(kParams * 4) || m->V.reserve(kParams * 4) ||
        m->loss.reserve(4)) {
      delete m;
      return fail(NGAP_ERR_OOM, "MLP allocation failed");
    }
    if (hipMemcpy(m->P.p, p.data(), kParams * 4, hipMemcpyHostToDevice) != hipSuccess) rc = 1;
    std::vector<float> zero(kParams, 0.f);
    if (hipMemcpy(m->M.p, zero.data(), kParams * 4, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(m->V.p, zero.data(), kParams * 4, hipMemcpyHostToDevice) != hipSuccess)
      rc = 1;
    if (rc) {
      delete m;
      return fail(NGAP_ERR_DEVICE, "MLP initialisation failed");
    }
    *out = m;
    return NGAP_OK;
  });
}

int ngap_mlp_destroy(ngap_mlp *m) {
  return ngapamd::c_guard([&]() -> int {
    delete m;
    return NGAP_OK;
  });
}

int32_t ngap_mlp_num_params(void) { return kParams; }

int ngap_mlp_get_params(ngap_mlp *m, float *out) {
  return ngapamd::c_guard([&]() -> int {
    if (!m || !out) return fail(NGAP_ERR_INVALID, "NULL argument");
    MLP_TRY(hipMemcpy(out, m->P.p, kParams * 4, hipMemcpyDeviceToHost));
    return NGAP_OK;
  });
}

int ngap_mlp_set_params(ngap_mlp *m, const float *in) {
  return ngapamd::c_guard([&]() -> int {
    if (!m || !in) return fail(NGAP_ERR_INVALID, "NULL argument");
    MLP_TRY(hipMemcpy(m->P.p, in, kParams * 4, hipMemcpyHostToDevice));
    return NGAP_OK;
  });
}

int ngap_mlp_predict(ngap_mlp *m, const float *x, uint64_t n, float *y) {
  return ngapamd::c_guard([&]() -> int {
    if (!m || (!x && n) || (!y && n)) return fail(NGAP_ERR_INVALID, "NULL argument");
    if (!n) return NGAP_OK;
    MLP_TRY(hipSetDevice(m->device));
    int rc = load_batch(m, x, nullptr, n);
    if (rc) return rc;
    MLP_TRY(m->Y.reserve(n * 4));
    hipLaunchKernelGGL(k_forward, dim3(blocks_for(n, kTile, 1024)), dim3(kThreads), 0, 0,
                       m->P.f(), m->X.f(), n, m->Y.f());
    MLP_TRY(hipGetLastError());
    MLP_TRY(hipMemcpy(y, m->Y.p, n * 4, hipMemcpyDeviceToHost));
    return NGAP_OK;
  });
}

int ngap_mlp_predict_pairs(ngap_mlp *m, const float *hist, uint32_t num_windows,
                           const float *stats, uint32_t num_groups, const uint32_t *pairs,
                           uint64_t n, float *y) {
  return ngapamd::c_guard([&]() -> int {
    if (!m || !hist || !stats || !pairs || !y) return fail(NGAP_ERR_INVALID, "NULL argument");
    if (!n) return NGAP_OK;
    if (!num_windows || !num_groups) return fail(NGAP_ERR_INVALID, "pair out of range");
    MLP_TRY(hipSetDevice(m->device));
    MLP_TRY(m->hist.reserve((size_t)num_windows * kHist * 4));
    MLP_TRY(m->stats.reserve((size_t)num_groups * 8 * 4));
    MLP_TRY(m->pairs.reserve(n * 8));
    MLP_TRY(m->Y.reserve(n * 4 + 4));
    MLP_TRY(m->parts.reserve(((size_t)num_windows + num_groups) * kHid * 4));
    MLP_TRY(hipMemcpy(m->hist.p, hist, (size_t)num_windows * kHist * 4, hipMemcpyHostToDevice));
    MLP_TRY(hipMemcpy(m->stats.p, stats, (size_t)num_groups * 8 * 4, hipMemcpyHostToDevice));
    MLP_TRY(hipMemcpy(m->pairs.p, pairs, n * 8, hipMemcpyHostToDevice));
    float *wpart = m->parts.f(), *gpart = wpart + (size_t)num_windows * kHid;
    uint32_t *bad = reinterpret_cast<uint32_t *>(m->Y.f() + n);  // set by a pair out of range
    const uint32_t wblocks = (num_windows + 15) / 16;
    hipLaunchKernelGGL(k_parts, dim3(wblocks + (num_groups + 15) / 16), dim3(256), 0, 0,
                       m->P.f(), m->hist.f(), num_windows, m->stats.f(), num_groups, wblocks,
                       wpart, gpart, bad);
    MLP_TRY(hipGetLastError());
    // three workgroups of 152 registers a lane fit each of 256 CUs; more would
    // run a second, partly empty turn (1,024: 190 us against 174)
    hipLaunchKernelGGL(k_pairs, dim3(blocks_for(n, 64, 768)), dim3(256), 0, 0, m->P.f(), wpart,
                       gpart, reinterpret_cast<uint2 *>(m->pairs.p), n, num_windows, num_groups,
                       m->Y.f(), bad);
    MLP_TRY(hipGetLastError());
    uint32_t wrong = 0;
    MLP_TRY(hipMemcpy(&wrong, bad, 4, hipMemcpyDeviceToHost));
    if (wrong) return fail(NGAP_ERR_INVALID, "pair out of range");
    MLP_TRY(hipMemcpy(y, m->Y.p, n * 4, hipMemcpyDeviceToHost));
    return NGAP_OK;
  });
}

int ngap_mlp_gradient(ngap_mlp *m, const float *x, const float *t, uint64_t n, float *grad,
                      float *loss) {
  return ngapamd::c_guard([&]() -> int {
    if (!m || !x || !t || !grad || !loss || !n) return fail(NGAP_ERR_INVALID, "bad argument");
    MLP_TRY(hipSetDevice(m->device));
    int rc = load_batch(m, x, t, n);
    if (rc) return rc;
    MLP_TRY(m->Y.reserve(kParams * 4));
    rc = grad_on_device(m, nullptr, n, m->Y.f(), m->loss.f(), Adam{});
    if (rc) return rc;
    MLP_TRY(hipMemcpy(grad, m->Y.p, kParams * 4, hipMemcpyDeviceToHost));
    float l = 0;
    MLP_TRY(hipMemcpy(&l, m->loss.p, 4, hipMemcpyDeviceToHost));
    *loss = l / (float)n;
    return NGAP_OK;
  });
}

int ngap_mlp_train(ngap_mlp *m, const float *x, const float *t, uint64_t n, int32_t epochs,
                   uint32_t batch, float lr, uint64_t seed, float *final_loss) {
  return ngapamd::c_guard([&]() -> int {
    if (!m || !x || !t || !n || epochs < 1 || batch < 1)
      return fail(NGAP_ERR_INVALID, "bad argument");
    MLP_TRY(hipSetDevice(m->device));
    // The samples stay on the device while they are trained on (up to
    // kResident bytes), and a mini-batch is a range of the epoch's shuffled
    // row numbers; beyond that each mini-batch is gathered on the host.
    const uint64_t steps = (n + batch - 1) / batch;  // per epoch
    MLP_TRY(m->loss.reserve(steps * 4));  // one sum per mini-batch of an epoch
    MLP_TRY(m->G.reserve(grad_bytes(std::min<uint64_t>(batch, n))));
    struct GiveBack {
      ngap_mlp *m;
      const size_t had;
      ~GiveBack() {
        if (m->X.n <= std::max<size_t>(had, kHeld)) return;
        m->X.release();
        m->T.release();
        m->idx.release();
      }
    } give_back{m, m->X.n};
    const bool resident = n < (1ull << 32) && n <= kResident / (kIn * 4) &&
                          m->X.reserve(n * kIn * 4) == hipSuccess &&
                          m->T.reserve(n * 4) == hipSuccess && m->idx.reserve(n * 4) == hipSuccess;
    if (!resident) (void)hipGetLastError();
    if (resident) {
      const int rc = load_batch(m, x, t, n);
      if (rc) return rc;
    }
    std::vector<uint32_t> rows32(resident ? n : 0);
    std::vector<uint64_t> rows64(resident ? 0 : n);
    std::vector<float> bx(resident ? 0 : (size_t)batch * kIn), bt(resident ? 0 : batch);
    for (uint64_t i = 0; i < rows32.size(); i++) rows32[i] = (uint32_t)i;
    for (uint64_t i = 0; i < rows64.size(); i++) rows64[i] = i;
    uint64_t z = seed;
    for (int e = 0; e < epochs; e++) {
      // (overlaps the last epoch's mini-batches when the samples are resident)
      for (uint64_t i = n - 1; i > 0; i--) {
        z = z * 6364136223846793005ull + 1442695040888963407ull;
        if (resident) std::swap(rows32[i], rows32[(uint32_t)(z >> 33) % (uint32_t)(i + 1)]);
        else std::swap(rows64[i], rows64[(z >> 33) % (i + 1)]);
      }
      if (resident) MLP_TRY(hipMemcpy(m->idx.p, rows32.data(), n * 4, hipMemcpyHostToDevice));
      for (uint64_t b0 = 0, k = 0; b0 < n; b0 += batch, k++) {
        const uint64_t nb = std::min<uint64_t>(batch, n - b0);
        if (!resident) {
          for (uint64_t i = 0; i < nb; i++) {
            memcpy(&bx[i * kIn], x + rows64[b0 + i] * kIn, kIn * 4);
            bt[i] = t[rows64[b0 + i]];
          }
          const int rc = load_batch(m, bx.data(), bt.data(), nb);
          if (rc) return rc;
        }
        m->step++;
        const float b1 = 0.9f, b2 = 0.999f;
        const Adam o{lr, b1, b2, 1e-8f, 1.f - std::pow(b1, (float)m->step),
                     1.f - std::pow(b2, (float)m->step)};
        const int rc = grad_on_device(
            m, resident ? reinterpret_cast<uint32_t *>(m->idx.p) + b0 : nullptr, nb, nullptr,
            m->loss.f() + k, o);
        if (rc) return rc;
      }
    }
    std::vector<float> sums(steps);
    MLP_TRY(hipMemcpy(sums.data(), m->loss.p, steps * 4, hipMemcpyDeviceToHost));
    double last = 0;
    for (float l : sums) last += l;
    last /= (double)n;
    if (final_loss) *final_loss = (float)last;
    return NGAP_OK;
  });
}

}  // extern "C"
